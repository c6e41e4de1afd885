// sqrt_sweep.hip -- st_sqrt (cookiedough_amd/csrc/ckd_sqrt.h) beside sqrtf on the
// device, for tests/test_gpu_sqrt.py.  One lane a mantissa; every index is below
// the 2^23 of its buffers, which the launch covers exactly.
#include "ckd_sqrt.h"

#include <cstdint>

namespace {
constexpr uint32_t kMantissas = 1u << 23, kBlock = 256;

__global__ __launch_bounds__(kBlock) void k_sweep(uint32_t exponent, uint32_t *__restrict__ out,
                                                  unsigned long long *__restrict__ differ)
{
    const uint32_t m = blockIdx.x * kBlock + threadIdx.x;
    const float x = __uint_as_float((exponent << 23) | m);
    const uint32_t got = __float_as_uint(st_sqrt(x));
    if (out) out[m] = got;
    if (got != __float_as_uint(sqrtf(x))) atomicAdd(differ, 1ull);
}
} // namespace

// all mantissas of the biased exponents first .. last: how many of st_sqrt's bits
// differ from sqrtf's, and (out, host, 2^23 words, may be null) st_sqrt's bits of
// the last exponent.  Negative: a HIP error.
extern "C" __attribute__((visibility("default"))) long long sqrt_sweep(uint32_t first, uint32_t last, uint32_t *out)
{
    if (first > last || last > 254) return -1;
    uint32_t *bits = nullptr;
    unsigned long long *differ = nullptr, n = 0;
    hipError_t e = hipMalloc(&differ, sizeof(n));
    if (e == hipSuccess && out) e = hipMalloc(&bits, kMantissas * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemcpy(differ, &n, sizeof(n), hipMemcpyHostToDevice);
    for (uint32_t x = first; x <= last && e == hipSuccess; ++x) {
        k_sweep<<<kMantissas / kBlock, kBlock>>>(x, x == last ? bits : nullptr, differ);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&n, differ, sizeof(n), hipMemcpyDeviceToHost);
    if (e == hipSuccess && out) e = hipMemcpy(out, bits, kMantissas * sizeof(uint32_t), hipMemcpyDeviceToHost);
    (void)hipFree(bits);
    (void)hipFree(differ);
    return e == hipSuccess ? (long long)n : -1;
}
