// identities.hip -- the device code's short forms of IEEE operations, compared
// with those operations over all their inputs (tests/test_gpu_identities.py).
// Built apart from the library; nothing but the test loads it.
#include <cstdint>

#include "../csrc/mh_device.hpp"

namespace {
using namespace mh;

constexpr uint32_t kBlocks = 4096, kThreads = 256;
enum { kTerms, kReciprocals, kQuotients, kChecks };

__device__ __forceinline__ bool differ(float a, float b) { return __float_as_uint(a) != __float_as_uint(b); }

__device__ __forceinline__ uint32_t mix(uint32_t x) {
    x = (x ^ x >> 16) * 0x7feb352du;
    x = (x ^ x >> 15) * 0x846ca68bu;
    return x ^ x >> 16;
}

// term_of_square against 1 / (sqrt(d) + 1) for the floats d whose bits are
// 0 to 0x7f800000 (infinity).
__global__ __launch_bounds__(kThreads) void terms_kernel(uint32_t* bad) {
    uint32_t n = 0;
    for (uint64_t u = blockIdx.x * kThreads + threadIdx.x; u <= 0x7f800000u; u += (uint64_t)kBlocks * kThreads) {
        const float d = __uint_as_float((uint32_t)u);
        n += differ(term_of_square(d), 1.0f / (sqrtf(d) + 1.0f)) ? 1u : 0u;
    }
    if (n) atomicAdd(bad + kTerms, n);
}

// div_unit for every b in (2^-60, 1]: 1 / b (its reciprocal is the first step's
// result), then quotients of a with 0 <= |a| <= b: both ends, neighbours of b,
// the smallest allowed and `pairs` of any mantissa and exponent between.
__global__ __launch_bounds__(kThreads) void divisions_kernel(uint32_t pairs, uint32_t* bad) {
    const uint32_t lo = 0x21800001u, hi = 0x3f800000u;  // 2^-60 (the next float), 1
    uint32_t nr = 0, nq = 0;
    for (uint64_t u = lo + blockIdx.x * kThreads + threadIdx.x; u <= hi; u += (uint64_t)kBlocks * kThreads) {
        const float b = __uint_as_float((uint32_t)u);
        float y = __builtin_amdgcn_rcpf(b);
        y = __builtin_fmaf(__builtin_fmaf(-b, y, 1.0f), y, y);
        nr += differ(y, 1.0f / b) ? 1u : 0u;
        uint32_t seed = (uint32_t)u;
        for (uint32_t i = 0; i < pairs + 4; ++i) {
            seed = mix(seed + 0x9e3779b9u);
            // an exponent from 2^-89 to b's, any mantissa; not above b
            const uint32_t eb = (uint32_t)u >> 23, e = 38u + seed % (eb - 37u);
            uint32_t a = e << 23 | mix(seed) >> 9;
            a = i == 0 ? (uint32_t)u : i == 1 ? (uint32_t)u - 1u : i == 2 ? 0x12800001u : i == 3 ? 0u : a;
            a = a > (uint32_t)u ? (uint32_t)u : a;
            const float q = __uint_as_float(a);
            nq += differ(div_unit(q, b), q / b) ? 1u : 0u;
            nq += a && differ(div_unit(-q, b), -q / b) ? 1u : 0u;
        }
    }
    if (nr) atomicAdd(bad + kReciprocals, nr);
    if (nq) atomicAdd(bad + kQuotients, nq);
}
}  // namespace

// out: the differing terms, reciprocals and quotients.  Returns the first HIP
// error.
extern "C" int mh_test_identities(uint32_t pairs, uint32_t* out) {
    uint32_t* bad = nullptr;
    hipError_t e = hipMalloc(&bad, kChecks * sizeof(uint32_t));
    if (e == hipSuccess) e = hipMemset(bad, 0, kChecks * sizeof(uint32_t));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(terms_kernel, dim3(kBlocks), dim3(kThreads), 0, nullptr, bad);
        hipLaunchKernelGGL(divisions_kernel, dim3(kBlocks), dim3(kThreads), 0, nullptr, pairs, bad);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, bad, kChecks * sizeof(uint32_t), hipMemcpyDeviceToHost);
    if (bad) (void)hipFree(bad);
    return (int)e;
}
