/*
 * hip_host.h -- the HIP runtime calls of the library's host code, on host
 * memory, for tests that run without a device: allocations are poisoned,
 * copies happen at once, and the n-th call can be made to fail.
 */
#ifndef HIP_HOST_H
#define HIP_HOST_H

#include <cstdint>
#include <cstdlib>
#include <cstring>

#include <hip/hip_runtime.h>

static long hip_calls = 0;          /* calls since hip_fail_at() */
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
}

#endif /* HIP_HOST_H */
