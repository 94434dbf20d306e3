// Random numbers of the event loop and the queue build.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace ssa {

// Philox4x32-10 (Salmon et al., SC'11) for the seeded stream.
__device__ __forceinline__ void philox(uint32_t c[4], uint32_t k0, uint32_t k1) {
    const uint32_t M0 = 0xD2511F53u, M1 = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
#pragma unroll
    for (int r = 0; r < 10; r++) {
        uint32_t hi0 = __umulhi(M0, c[0]), lo0 = M0 * c[0];
        uint32_t hi1 = __umulhi(M1, c[2]), lo1 = M1 * c[2];
        uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
        k0 += W0; k1 += W1;
    }
}
__device__ __forceinline__ uint64_t philox64(uint64_t seed, uint64_t stream, uint64_t ctr) {
    uint32_t c[4] = {(uint32_t)ctr, (uint32_t)(ctr >> 32), (uint32_t)stream, (uint32_t)(stream >> 32)};
    philox(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    return (uint64_t)c[0] | ((uint64_t)c[1] << 32);
}
// rng()*1.0/rng.max() (simulate_rdme.cpp:253, 353); the divisor is 2^64 as a
// double, so this is also generate_canonical's value
__device__ __forceinline__ double word_uniform(uint64_t w) {
    return (double)w * 1.0 / (double)0xFFFFFFFFFFFFFFFFULL;
}
// -log(1 - generate_canonical) (libstdc++ exponential_distribution) of a
// word's uniform value
__device__ __forceinline__ double uniform_expo(double u) {
    double c = u;
    if (c >= 1.0) c = 0x1.fffffffffffffp-1;
    return -log(1.0 - c) / 1.0;
}
__device__ __forceinline__ double word_expo(uint64_t w) { return uniform_expo(word_uniform(w)); }

}  // namespace ssa
