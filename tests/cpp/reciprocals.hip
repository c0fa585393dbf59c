// recip() of the triangular kernels against the division, for every significand at the exponents first .. last, on the device. Run by
// tests/test_gpu_reciprocals.py.
#include "rmx_tri_math.h"

constexpr uint32_t SIGNIFICANDS = 1u << 23;

__global__ void __launch_bounds__(256) reciprocals(int first, int last, unsigned long long *wrong, unsigned long long *seen) {
    unsigned long long w = 0, n = 0;
    for (uint32_t m = blockIdx.x * 256 + threadIdx.x; m < SIGNIFICANDS; m += gridDim.x * 256)
        for (int e = first; e <= last; e++) {
            const float b = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23 | m);
            w += __builtin_bit_cast(uint32_t, rmx::recip(b)) != __builtin_bit_cast(uint32_t, 1.0f / b);
            n++;
        }
    atomicAdd(wrong, w);
    atomicAdd(seen, n);
}

// counts: two 64-bit numbers in device memory, cleared: values that differ, values compared
extern "C" __attribute__((visibility("default"))) int reciprocals_check(int first, int last, void *counts, void *stream) {
    if (first < -126 || last > 126 || first > last || !counts) return -1;
    unsigned long long *c = static_cast<unsigned long long *>(counts);
    hipLaunchKernelGGL(reciprocals, dim3(2048), dim3(256), 0, static_cast<hipStream_t>(stream), first, last, c, c + 1);
    return (int)hipGetLastError();
}
