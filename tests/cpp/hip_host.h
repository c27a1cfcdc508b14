/*
 * hip_host.h -- the HIP runtime calls of the library's host code, on host
 * memory, for tests that run without a device: allocations are poisoned,
 * copies happen at once, and the n-th call can be made to fail.
 */
#ifndef HIP_HOST_H
#define HIP_HOST_H

#include <atomic>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#include <hip/hip_runtime.h>

static std::atomic<long> hip_calls{0};  /* calls since hip_fail_at() */
static long hip_fail_on = -1;       /* the call that fails, -1: none */

static void hip_fail_at(long n)
{
    hip_calls = 0;
    hip_fail_on = n;
}
static hipError_t hip_step(hipError_t as = hipErrorUnknown)
{
    return hip_calls++ == hip_fail_on ? as : hipSuccess;
}
static hipError_t hip_get(void **p, size_t n)
{
    *p = nullptr;
    if (hip_step() != hipSuccess) return hipErrorOutOfMemory;
    *p = malloc(n);
    memset(*p, 0xA5, n);
    return hipSuccess;
}

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { return hip_get(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hip_get(p, n); }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    *e = (hipEvent_t)malloc(1);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hip_step(); }
hipError_t hipEventSynchronize(hipEvent_t) { return hip_step(); }
hipError_t hipStreamSynchronize(hipStream_t) { return hip_step(); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    return hipMemcpyAsync(d, s, n, k, nullptr);
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "failed on purpose"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    if (hip_step() != hipSuccess) return hipErrorUnknown;
    *s = (hipStream_t)malloc(1);
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamDestroy(hipStream_t s) { free((void *)s); return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorUnknown; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorUnknown; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return hipErrorUnknown;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorUnknown; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

#endif /* HIP_HOST_H */
