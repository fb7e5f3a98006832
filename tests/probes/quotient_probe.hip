// quotient_probe.hip -- checks, on the GPU, the FP64 sequences of the step kernels with the kernels'
// own functions (shll_device.h), on random positive doubles:
//   quot(a, b, rcp_nr2(b))             == a / b        (F64's primitives)
//   sqrt_rcp(x, s, y): s               == sqrt(x), and quot(a, s, y) == a / s
//   rsq_sqrt(x, y, s): s               within a stated number of ulp of sqrt(x)  (F64F)
// The right-hand sides are the IEEE operators.
// Test infrastructure: loaded only by tests/test_gpu_quotients.py.
#include <stdint.h>

#include "shll_device.h"

namespace {

__device__ __forceinline__ uint64_t mix64(uint64_t x) {  // SplitMix64 finaliser
    x += 0x9e3779b97f4a7c15ull;
    x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
    x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
    return x ^ (x >> 31);
}

// mantissa uniform, exponent in [-span, span]
__device__ __forceinline__ double random_double(uint64_t h, int span) {
    const uint64_t e = (uint64_t)((int)(mix64(h ^ 0x5851f42d4c957f2dull) % (uint64_t)(2 * span + 1)) - span + 1023);
    return __longlong_as_double((long long)(e << 52 | (h & 0xfffffffffffffull)));
}

__device__ __forceinline__ bool differ(double a, double b) { return __double_as_longlong(a) != __double_as_longlong(b); }

// out[0..2]: mismatches of the quotient, the root, the quotient by the root; out[3]: ulp of rsq_sqrt's root
__global__ void k_check(unsigned long long* out, int reps, uint64_t seed) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long c[3] = {0, 0, 0};
    long long ulp = 0;
    for (int i = 0; i < reps; ++i) {
        const uint64_t h = mix64((t * (uint64_t)reps + (uint64_t)i) * 4ull + seed);
        const double a = random_double(mix64(h), 200), b = random_double(mix64(h + 1), 200);
        c[0] += differ(shll::quot(a, b, shll::rcp_nr2(b)), a / b);
        double s, y;
        shll::sqrt_rcp(b, s, y);
        c[1] += differ(s, sqrt(b));
        c[2] += differ(shll::quot(a, s, y), a / sqrt(b));
        const double x = random_double(mix64(h + 2), 1000);
        shll::rsq_sqrt(x, y, s);
        long long d = __double_as_longlong(s) - __double_as_longlong(sqrt(x));
        d = d < 0 ? -d : d;
        ulp = d > ulp ? d : ulp;
    }
    for (int q = 0; q < 3; ++q)
        if (c[q]) atomicAdd(&out[q], c[q]);
    if (ulp) atomicMax(&out[3], (unsigned long long)ulp);
}

}  // namespace

// 2^20 * reps arguments; 0 or a HIP error
extern "C" int probe_quotients(int reps, unsigned long long seed, unsigned long long* out) {
    unsigned long long* d = nullptr;
    hipError_t e = hipMalloc((void**)&d, 4 * sizeof(*d));
    if (e != hipSuccess) return (int)e;
    for (int q = 0; q < 4; ++q) out[q] = 0;
    e = hipMemcpy(d, out, 4 * sizeof(*d), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_check, dim3((1 << 20) / 256), dim3(256), 0, 0, d, reps, (uint64_t)seed);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, d, 4 * sizeof(*d), hipMemcpyDeviceToHost);
    (void)hipFree(d);
    return (int)e;
}
