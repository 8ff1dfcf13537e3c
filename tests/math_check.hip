// math_check.hip -- the short reciprocals and quotients of hr_math.h against
// the compiler's correctly rounded division, on the GPU.  Built with the
// library's flags into tests/libmath_check.so; test_gpu_math.py runs it.
#include "hr_math.h"

namespace {

using namespace hr;

__device__ bool same(float a, float b)
{
    return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
}

// bad: {count, operands of one mismatch}
__device__ void report(unsigned long long* bad, float a, float b)
{
    atomicAdd(bad, 1ull);
    bad[1] = (unsigned long long)__float_as_uint(a) << 32 | __float_as_uint(b);
}

// every float: rcp_rn, and rcp_in_range where it is declared
__global__ void k_rcp(unsigned long long* bad)
{
    const uint64_t n = 1ull << 32;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const float x = __uint_as_float((uint32_t)i);
        const float want = 1.f / x;
        if (!same(rcp_rn(x), want)) report(bad, x, rcp_rn(x));
        const float a = fabsf(x);
        if (a >= kRcpLow && a <= kRcpHigh && !same(rcp_in_range(x), want)) report(bad, x, rcp_in_range(x));
    }
}

__device__ void check_div(unsigned long long* bad, float a, float b)
{
    const float q = div_by_rcp(a, b, rcp_rn(b)), want = a / b;
    if (!same(q, want) && !(a == 0.f && q == want)) report(bad, a, b);      // the sign of a zero is not kept
}

__device__ float make(uint32_t sign, int e, uint32_t m)
{
    return __uint_as_float(sign << 31 | (uint32_t)(e + 127) << 23 | (m & 0x7FFFFFu));
}

// significands where roundings turn: about 1, 1.5, 2, the square root of 2 and thirds
__device__ uint32_t corner(uint32_t i)
{
    const uint32_t base[8] = { 0u, 0x400000u, 0x800000u, 0x3504F3u, 0x2AAAAAu, 0x555555u, 0x200000u, 0x600000u };
    return (base[i >> 4 & 7u] + (i & 15u) - 8u) & 0x7FFFFFu;
}

// all pairs of 128 corner significands, exponents at the ends of the range and
// in the middle, both signs, and numerators of zero
__global__ void k_div_corners(unsigned long long* bad)
{
    const int ex[7] = { -60, -59, -1, 0, 1, 58, 59 };
    const uint32_t ia = blockIdx.x, ib = threadIdx.x;
    for (int p = 0; p < 7; ++p)
        for (int q = 0; q < 7; ++q)
            for (uint32_t s = 0; s < 4; ++s) check_div(bad, make(s & 1u, ex[p], corner(ia)), make(s >> 1, ex[q], corner(ib)));
    for (int q = 0; q < 7; ++q)
        for (uint32_t s = 0; s < 4; ++s) check_div(bad, s & 1u ? -0.f : 0.f, make(s >> 1, ex[q], corner(ib)));
    for (uint32_t s = 0; s < 4; ++s)                                 // the bounds themselves
        for (int p = -1; p < 7; ++p) {
            check_div(bad, p < 0 ? 0x1p60f : make(s & 1u, ex[p], corner(ia)), s >> 1 ? -0x1p60f : 0x1p60f);
            check_div(bad, s & 1u ? -0x1p60f : 0x1p60f, p < 0 ? -0x1p60f : make(s >> 1, ex[p], corner(ib)));
        }
}

__device__ uint64_t mix(uint64_t z)         // SplitMix64 (Steele, Lea and Flood, OOPSLA 2014)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ z >> 30) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ z >> 27) * 0x94D049BB133111EBull;
    return z ^ z >> 31;
}

__global__ void k_div_random(unsigned long long* bad, uint64_t n, uint64_t seed)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t u = mix(seed + i), v = mix(~seed - i);
        check_div(bad, make((uint32_t)(u >> 63), (int)((u >> 32 & 0xFFFFu) % 120u) - 60, (uint32_t)u),
                  make((uint32_t)(v >> 63), (int)((v >> 32 & 0xFFFFu) % 120u) - 60, (uint32_t)v));
    }
}

}  // namespace

// what: 0 reciprocals of every float, 1 corner quotients, 2 n random quotients.
// out: mismatches and one pair of operands.  Returns a hipError_t.
extern "C" int math_check(int what, unsigned long long n, unsigned long long seed, unsigned long long* out)
{
    unsigned long long* bad = nullptr;
    hipError_t e = hipMalloc((void**)&bad, 2 * sizeof *bad);
    if (e != hipSuccess) return (int)e;
    e = hipMemset(bad, 0, 2 * sizeof *bad);
    if (what == 0) hipLaunchKernelGGL(k_rcp, dim3(4096), dim3(256), 0, nullptr, bad);
    else if (what == 1) hipLaunchKernelGGL(k_div_corners, dim3(128), dim3(128), 0, nullptr, bad);
    else hipLaunchKernelGGL(k_div_random, dim3(4096), dim3(256), 0, nullptr, bad, (uint64_t)n, (uint64_t)seed);
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpy(out, bad, 2 * sizeof *bad, hipMemcpyDeviceToHost);
    const hipError_t f = hipFree(bad);
    return (int)(e != hipSuccess ? e : f);
}
