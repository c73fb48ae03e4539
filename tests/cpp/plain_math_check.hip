// The quotients and roots of the Jacobi pairs (plain_root, refined_rcp and plain_quotient in mpm_math.hpp) against
// double: every float they can meet where that is one float, sampled pairs where it is two.  A float
// quotient or root is the double one rounded (53 >= 2 * 24 + 2 bits).
#include <hip/hip_runtime.h>

#include "../../nuclearmpm_amd/csrc/mpm_math.hpp"

namespace {

using namespace nclr_dev;

__device__ bool same(float a, float b) { return __float_as_uint(a) == __float_as_uint(b); }

__device__ uint32_t mix(uint64_t x) {  // splitmix64
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return uint32_t((x ^ (x >> 31)) >> 16);
}

__device__ bool quotient_ok(float n, float d) {
    return same(plain_quotient(n, d, refined_rcp(d)), float(double(n) / double(d)));
}

// counts[2 c] cases checked and counts[2 c + 1] of them wrong, by check c:
//   0  plain_root, both parts, for every float of [1, 2^90]
//   1  refined_rcp twice for every float of [1, 2^44] and (-2^44, -1]
//   2  plain_quotient(u, sqrt(1 + u^2)) from plain_root's reciprocal, |u| every float of [2^-43, 2^43]
//   3  plain_quotient from refined_rcp: every significand of the denominator, numerators at random and next to
//      the products of the denominator with midpoints between floats, where rounding is decided last
__global__ __launch_bounds__(256) void k_check(unsigned long long* counts) {
    const uint64_t threads = uint64_t(gridDim.x) * blockDim.x, t0 = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    unsigned long long n[4] = {}, bad[4] = {};
    for (uint64_t b = 0x3F800000u + t0; b <= 0x3F800000u + 90ull * (1u << 23); b += threads) {
        const float x = __uint_as_float(uint32_t(b));
        const Root r = plain_root(x);
        float y;
        const float s = float(sqrt(double(x)));
        ++n[0];
        bad[0] += !(same(plain_root(x, y), s) && same(r.s, s) && same(r.r, float(1.0 / double(s))));
    }
    for (uint64_t b = 0x3F800000u + t0; b <= 0x3F800000u + 44ull * (1u << 23); b += threads)
        for (uint32_t sign = 0; sign < 2; ++sign) {
            const float v = __uint_as_float(uint32_t(b) | sign << 31);
            ++n[1];
            bad[1] += !same(refined_rcp(v, refined_rcp(v)), float(1.0 / double(v)));
        }
    for (uint64_t b = 0x3F800000u - 43ull * (1u << 23) + t0; b <= 0x3F800000u + 43ull * (1u << 23); b += threads)
        for (uint32_t sign = 0; sign < 2; ++sign) {
            const float u = __uint_as_float(uint32_t(b) | sign << 31);
            const Root r = plain_root(1.0f + u * u);
            ++n[2];
            bad[2] += !same(plain_quotient(u, r.s, r.r), float(double(u) / double(r.s)));
        }
    for (uint64_t m = t0; m < (1u << 23); m += threads)
        for (uint32_t k = 0; k < 64; ++k) {
            const uint32_t h = mix(m * 64 + k), g = mix(~(m * 64 + k));
            // exponents of d and n in [-40, 40], any signs
            const float d = __uint_as_float(uint32_t(m) | (127u - 40u + h % 80u) << 23 | (h & 0x80000000u));
            const float a = __uint_as_float((g & 0x7FFFFFu) | (127u - 40u + (g >> 8) % 80u) << 23 | (g & 0x80000000u));
            ++n[3];
            bad[3] += !quotient_ok(a, d);
            // next to d times a midpoint q + half a unit, q in [1, 2)
            const double mid = 1.0 + (double(g & 0x7FFFFFu) + 0.5) * 0x1p-23;
            const uint32_t e = __float_as_uint(float(double(d) * mid));
            for (int o = -1; o <= 1; ++o) {
                ++n[3];
                bad[3] += !quotient_ok(__uint_as_float(e + uint32_t(o)), d);
            }
        }
    for (int c = 0; c < 4; ++c) {
        atomicAdd(&counts[2 * c], n[c]);
        atomicAdd(&counts[2 * c + 1], bad[c]);
    }
}

}  // namespace

// host: eight words, counts as above.  0 or a hipError_t.
extern "C" int plain_math_check(unsigned long long* host) {
    unsigned long long* counts = nullptr;
    hipError_t e = hipMalloc(reinterpret_cast<void**>(&counts), 8 * sizeof(*counts));
    if (e != hipSuccess) return int(e);
    for (int c = 0; c < 8; ++c) host[c] = 0;
    e = hipMemcpy(counts, host, 8 * sizeof(*counts), hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        k_check<<<4096, 256>>>(counts);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(host, counts, 8 * sizeof(*counts), hipMemcpyDeviceToHost);
    (void)hipFree(counts);
    return int(e);
}
