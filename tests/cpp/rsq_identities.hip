// The square root and the reciprocals of the fluid terms (cn_device.h fsqrt_rsq, fsqrt_nearzero_free,
// frcp_exact, frcp_exact_ge1), which refine this chip's estimates by one step, against the correctly
// rounded values: every significand at every exponent from 2^-96 to 2^98 (the root and its reciprocal)
// and from 2^-48 to 2^125 (the reciprocals).  Returns 0 when all agree.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "../../cressim-neo_amd/csrc/cn_device.h"

using namespace cn;

__global__ void check_root(uint32_t base, unsigned long long *bad)
{
    const float x = __uint_as_float(base + blockIdx.x * blockDim.x + threadIdx.x);
    const double root = sqrt((double)x);
    float y, z;
    const float s = fsqrt_rsq(x, y), t = fsqrt_nearzero_free(x, z), want = (float)root;
    // a double's root or quotient lies too far from a float's midpoint for a second rounding to matter
    const bool ok = s == want && t == want && frcp_exact(s, y) == (float)(1.0 / (double)want);
    if (!ok) atomicAdd(bad, 1ull);
}

__global__ void check_reciprocal(uint32_t base, unsigned long long *bad)
{
    const float b = __uint_as_float(base + blockIdx.x * blockDim.x + threadIdx.x);
    const float want = (float)(1.0 / (double)b);
    const bool ok = frcp_exact(b, __builtin_amdgcn_rcpf(b)) == want && (b < 1.0f || frcp_exact_ge1(b) == want);
    if (!ok) atomicAdd(bad, 1ull);
}

int main()
{
    unsigned long long *bad = nullptr, host = 0, total = 0;
    if (hipMalloc(&bad, sizeof(host)) != hipSuccess) return 2;
    const dim3 grid((1u << 23) / 256u), block(256);
    for (int e = -96; e <= 125; ++e) {
        if (hipMemset(bad, 0, sizeof(host)) != hipSuccess) return 2;
        const uint32_t base = (uint32_t)(127 + e) << 23;
        if (e <= 98) hipLaunchKernelGGL(check_root, grid, block, 0, 0, base, bad);
        if (e >= -48) hipLaunchKernelGGL(check_reciprocal, grid, block, 0, 0, base, bad);
        if (hipMemcpy(&host, bad, sizeof(host), hipMemcpyDeviceToHost) != hipSuccess) return 2;
        if (host) std::printf("exponent %d: %llu wrong\n", e, host);
        total += host;
    }
    (void)hipFree(bad);
    if (total == 0) std::printf("checks passed\n");
    return total ? 1 : 0;
}
