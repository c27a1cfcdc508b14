/*
 * device_math.hip -- the short forms of tracer_dev.h against fp64, on every
 * float: roots and reciprocal roots (a correctly rounded fp32 root or
 * quotient is the fp64 one rounded once more), texel channels, and the test
 * that keeps roots in the ray's range.
 */
#include "tracer_dev.h"

namespace {

enum { SQRT_MID, ROOT, RSQ, UNORM8, NEAR_T0, NEAR, N_BAD };
constexpr unsigned BLOCKS = 4096, WG = 256;

__device__ bool same(float a, float b)
{
    return fbits(a) == fbits(b) || (a != a && b != b);
}

/* every float, the waves' 64 neighbours apart by "step" of the index's bits:
 * 1 keeps a wave's values together (the short forms), an odd number mixes
 * them with values the short forms are not for */
__global__ void __launch_bounds__(WG) k_roots(uint32_t step, unsigned long long *bad)
{
    for (uint64_t i = blockIdx.x * (uint64_t)WG + threadIdx.x; i < 1ull << 32;
         i += (uint64_t)BLOCKS * WG)
    {
        const float x = bitsf((uint32_t)i * step);
        const float s = (float)sqrt((double)x);
        const float q = (float)(1.0 / (double)s);
        if (!same(root(x), s)) atomicAdd(&bad[ROOT], 1ull);
        if (!same(rsq(x), q)) atomicAdd(&bad[RSQ], 1ull);
        if (x == 0.0f || x >= SQRT_MID_MIN)
        {
            if (!same(sqrt_mid(x), s)) atomicAdd(&bad[SQRT_MID], 1ull);
        }
    }
}

__global__ void k_unorm8(unsigned long long *bad)
{
    const uint32_t c = threadIdx.x;
    if (!same(unorm8(c), (float)((double)c / 255.0))) atomicAdd(&bad[UNORM8], 1ull);
}

__device__ uint32_t mix(uint64_t &s)
{
    s = s * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(s >> 33) * 2654435761u ^ (uint32_t)(s >> 29);
}
/* a float of any bits, of a middle exponent, or a limit of the range */
__device__ float any_float(uint64_t &s)
{
    const uint32_t r = mix(s), k = mix(s) % 8;
    if (k == 0) return bitsf(r);
    if (k == 1) return bitsf((r & 0x80000003u) | ((r >> 8) % 3 == 0 ? 0x7f7ffffcu : 0u));
    return bitsf((r & 0x80ffffffu) | 0x3f000000u) * (k < 4 ? 1.0f : 1024.0f);
}

/* no root that the walk would take is turned away: t = n / d with
 * t_min < t <= t_lim, near values of t_min and t_lim among them */
__global__ void __launch_bounds__(WG) k_near(unsigned long long *bad)
{
    uint64_t s = (blockIdx.x * (uint64_t)WG + threadIdx.x) * 0x9e3779b97f4a7c15ull + 1u;
    for (int k = 0; k < 512; k++)
    {
        const float n = any_float(s), d = any_float(s);
        const float t = n / d;
        float t_min = fabsf(any_float(s)), t_lim = fabsf(any_float(s));
        const uint32_t pick = mix(s);
        if (pick & 1u) t_lim = bitsf(fbits(t) + (pick >> 8) % 3);
        if (pick & 2u) t_min = bitsf(fbits(t) - 1u - (pick >> 16) % 2);
        if (pick & 4u) t_min = -t_min;
        /* (the limit is the float below the ray's t_max, or a kept distance) */
        if (!(t_lim < INFINITY)) t_lim = 3.402823466e+38f;
        const bool near = in_lane(roots_near<false>(n, d, t_min, above<false>(t_lim)));
        if (t_min < t && t <= t_lim && !near) atomicAdd(&bad[NEAR], 1ull);
        const bool near0 = in_lane(roots_near<true>(n, d, 0.0f, above<true>(t_lim)));
        if (0.0f < t && t <= t_lim && !near0) atomicAdd(&bad[NEAR_T0], 1ull);
    }
}

} /* namespace */

/* counts of wrong results into bad[N_BAD]; 0, or a runtime error's code */
extern "C" int qrcheck_math(unsigned long long *bad)
{
    unsigned long long *dev = nullptr;
    hipError_t e = hipMalloc((void **)&dev, sizeof(*bad) * N_BAD);
    if (e != hipSuccess) return (int)e;
    e = hipMemset(dev, 0, sizeof(*bad) * N_BAD);
    if (e == hipSuccess)
    {
        hipLaunchKernelGGL(k_roots, dim3(BLOCKS), dim3(WG), 0, nullptr, 1u, dev);
        hipLaunchKernelGGL(k_roots, dim3(BLOCKS), dim3(WG), 0, nullptr, 2654435761u, dev);
        hipLaunchKernelGGL(k_unorm8, dim3(1), dim3(WG), 0, nullptr, dev);
        hipLaunchKernelGGL(k_near, dim3(BLOCKS), dim3(WG), 0, nullptr, dev);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(bad, dev, sizeof(*bad) * N_BAD, hipMemcpyDeviceToHost);
    (void)hipFree(dev);
    return (int)e;
}
