// The device's fp32 -> bf16 narrowing (common.h: f32x2_to_bf16, f32_to_bf16_ref) against its definition in integer steps (bf16_convert.h, which
// tests/bf16_exhaustive.cpp holds against the oracle's), over all 2^32 bit patterns, in either half of a pair.
// Built with the libraries; run by tests/test_bf16_narrowing_gpu.py; prints the number of mismatches of each.
#include <stdio.h>

#include "common.h"

using namespace xfthip;

// grid 4096 x 256 threads, 4096 patterns each; a pattern's neighbour in the pair is one that is not near it
__global__ __launch_bounds__(256) void sweep_kernel(unsigned long long *bad) {
    const uint32_t first = (blockIdx.x * 256u + threadIdx.x) * 4096u;
    unsigned lo = 0, hi = 0, one = 0;
    for (uint32_t i = 0; i < 4096u; ++i) {
        const uint32_t u = first + i, other = u * 2654435761u;
        const uint32_t want = f32_bits_to_bf16_ref(u), beside = f32_bits_to_bf16_ref(other);
        lo += f32x2_to_bf16(u2f(u), u2f(other)) != (want | beside << 16);
        hi += f32x2_to_bf16(u2f(other), u2f(u)) != (beside | want << 16);
        one += f32_to_bf16_ref(u2f(u)) != want;
    }
    if (lo) atomicAdd(bad, (unsigned long long)lo);
    if (hi) atomicAdd(bad + 1, (unsigned long long)hi);
    if (one) atomicAdd(bad + 2, (unsigned long long)one);
}

int main() {
    unsigned long long *dev = nullptr, bad[3] = {1, 1, 1};
    bool ok = hipMalloc((void **)&dev, sizeof(bad)) == hipSuccess && hipMemset(dev, 0, sizeof(bad)) == hipSuccess;
    if (ok) hipLaunchKernelGGL(sweep_kernel, dim3(4096), dim3(256), 0, 0, dev);
    ok = ok && hipGetLastError() == hipSuccess && hipMemcpy(bad, dev, sizeof(bad), hipMemcpyDeviceToHost) == hipSuccess;
    if (dev) (void)hipFree(dev);
    printf("%s lo=%llu hi=%llu one=%llu\n", ok ? "mismatches" : "failed", bad[0], bad[1], bad[2]);
    return ok && !(bad[0] | bad[1] | bad[2]) ? 0 : 1;
}
