// The unscaled reciprocal, quotient and square root of cn_math.h against the
// device's own IEEE operators, on the device (tests/test_gpu_device_math.py).
// Each call counts the operands that give other bits and hands back one.

#include <hip/hip_runtime.h>

#include "cn_math.h"

namespace {

using namespace cn;

constexpr uint32_t BLOCKS = 2048, THREADS = 256;

__device__ void compare(float got, float want, uint32_t a, uint32_t b, unsigned long long* result) {
    if (__float_as_uint(got) == __float_as_uint(want) || (isnan(got) && isnan(want))) return;
    if (atomicAdd(&result[0], 1ull) == 0) result[1] = uint64_t(a) << 32 | b;
}

// Every float whose bits lie in [first, last], of both signs for the reciprocal.
__global__ __launch_bounds__(THREADS) void k_every(int root, uint32_t first, uint32_t last,
                                                   unsigned long long* result) {
    for (uint64_t u = first + uint64_t(blockIdx.x) * THREADS + threadIdx.x; u <= last; u += uint64_t(BLOCKS) * THREADS) {
        const float x = __uint_as_float(uint32_t(u));
        if (root) {
            compare(sqrt_n(x), sqrtf(x), uint32_t(u), 0, result);
        } else {
            compare(rcp_n(x), 1.0f / x, uint32_t(u), 0, result);
            compare(rcp_n(-x), 1.0f / -x, uint32_t(u) | 0x80000000u, 0, result);
        }
    }
}

__device__ uint32_t mix(uint64_t v) {  // SplitMix64's finalizer
    v = (v ^ v >> 30) * 0xbf58476d1ce4e5b9ull;
    v = (v ^ v >> 27) * 0x94d049bb133111ebull;
    return uint32_t((v ^ v >> 31) >> 16);
}

// `count` quotients of random operands: a divisor of exponent -126 to 124, a
// dividend and a quotient of exponent -99 to 125, both of either sign; every
// fourth mantissa one of the first or the last 16.
__global__ __launch_bounds__(THREADS) void k_quotients(uint64_t seed, uint64_t count, unsigned long long* result) {
    for (uint64_t i = uint64_t(blockIdx.x) * THREADS + threadIdx.x; i < count; i += uint64_t(BLOCKS) * THREADS) {
        const uint32_t r0 = mix(seed + 4 * i), r1 = mix(seed + 4 * i + 1), r2 = mix(seed + 4 * i + 2),
                       r3 = mix(seed + 4 * i + 3);
        const auto mantissa = [](uint32_t r, uint32_t kind) {
            const uint32_t m = r & 0x7fffffu;
            return kind ? m : (m & 16u ? 0x7fffffu - (m & 15u) : m & 15u);
        };
        const int eb = int(r2 % 251) - 126;
        // a's exponent, so that its own and the quotient's (within one of the difference) stay in range
        const int lo = eb < 0 ? -99 : min(eb - 98, 125), hi = eb < 0 ? max(eb + 124, -99) : 125;
        if (lo > hi) continue;
        const int ea = lo + int(r3 % uint32_t(hi - lo + 1));
        const uint32_t a = (r0 & 0x80000000u) | uint32_t(ea + 127) << 23 | mantissa(r0, r3 >> 20 & 3u);
        const uint32_t b = (r1 & 0x80000000u) | uint32_t(eb + 127) << 23 | mantissa(r1, r3 >> 22 & 3u);
        const float fa = __uint_as_float(a), fb = __uint_as_float(b);
        const float want = fa / fb;
        if (!(fabsf(want) >= 0x1p-100f && fabsf(want) <= 0x1p126f)) continue;
        compare(div_n(fa, fb), want, a, b, result);
    }
}

// Runs `launch(result)` on zeroed counters and hands them back.
template <typename Launch>
int run(unsigned long long* out, Launch&& launch) {
    unsigned long long* result = nullptr;
    if (hipMalloc(reinterpret_cast<void**>(&result), 16) != hipSuccess) return 1;
    hipError_t e = hipMemset(result, 0, 16);
    if (e == hipSuccess) {
        launch(result);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(out, result, 16, hipMemcpyDeviceToHost);
    (void)hipFree(result);
    return e == hipSuccess ? 0 : 1;
}

}  // namespace

extern "C" {

int device_math_every(int root, uint32_t first, uint32_t last, unsigned long long* out) {
    return run(out, [&](unsigned long long* result) {
        hipLaunchKernelGGL(k_every, dim3(BLOCKS), dim3(THREADS), 0, nullptr, root, first, last, result);
    });
}

int device_math_quotients(uint64_t seed, uint64_t count, unsigned long long* out) {
    return run(out, [&](unsigned long long* result) {
        hipLaunchKernelGGL(k_quotients, dim3(BLOCKS), dim3(THREADS), 0, nullptr, seed, count, result);
    });
}

}  // extern "C"
