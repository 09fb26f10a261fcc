// Device std::mt19937 (the engine of ompl::RNG, util/RandomNumbers.h:190) and
// libstdc++'s generate_canonical<double, 53> over it (the 0-1 distribution
// of RNG::uniformReal, util/RandomNumbers.h:72-76, :191).
//
// The 624-word state lives in LDS.  The in-place recurrence
//   new[i] = src[i+397] ^ twist(old[i], old[i+1])   (indices mod 624)
// reads src from the new words from i = 227 on: new[i] then needs new[i-227].
// So the chain t, t+227, t+454 depends on no other chain: one thread computes
// it from old words alone, the block needs no barrier within a twist, and only
// word 623 wants a word of another chain (new[0]), which it makes again.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ompl_amd {

constexpr int kMtN = 624;
constexpr int kMtM = 397;
constexpr uint32_t kMtMatrix = 0x9908b0dfu;
constexpr uint32_t kMtUpper = 0x80000000u, kMtLower = 0x7fffffffu;

__device__ __forceinline__ uint32_t mt_twist_word(uint32_t cur, uint32_t next, uint32_t src)
{
    const uint32_t y = (cur & kMtUpper) | (next & kMtLower);
    return src ^ (y >> 1) ^ ((y & 1u) ? kMtMatrix : 0u);
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t y)
{
    y ^= y >> 11;
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= y >> 18;
    return y;
}

// std::mt19937::seed(v) by one thread (the recurrence is serial).
__device__ __forceinline__ void mt_seed_serial(uint32_t *mt, uint32_t v)
{
    mt[0] = v;
    for (int i = 1; i < kMtN; ++i) {
        v = 1812433253u * (v ^ (v >> 30)) + (uint32_t)i;
        mt[i] = v;
    }
}

// Twist of the LDS state by the whole block (at least 64 threads; every thread
// must call it): every old word is read before any new one is written, two
// barriers in all.
__device__ __forceinline__ void mt_twist_block(uint32_t *mt)
{
    constexpr int kChains = 227, kMost = (kChains + 63) / 64;
    uint32_t v[kMost][3];
#pragma unroll
    for (int i = 0; i < kMost; ++i) {
        const int t = threadIdx.x + i * blockDim.x;
        if (t < kChains) {
            v[i][0] = mt_twist_word(mt[t], mt[t + 1], mt[t + kMtM]);
            v[i][1] = mt_twist_word(mt[t + 227], mt[t + 228], v[i][0]);
            if (t < 169) v[i][2] = mt_twist_word(mt[t + 454], mt[t + 455], v[i][1]);
            else if (t == 169) v[i][2] = mt_twist_word(mt[623], mt_twist_word(mt[0], mt[1], mt[kMtM]), v[i][1]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMost; ++i) {
        const int t = threadIdx.x + i * blockDim.x;
        if (t < kChains) {
            mt[t] = v[i][0];
            mt[t + 227] = v[i][1];
            if (t < 170) mt[t + 454] = v[i][2];
        }
    }
    __syncthreads();
}

// generate_canonical<double, 53> from two tempered words (w1 first):
// (w1 + w2 * 2^32) / 2^64; a value rounding to 1 becomes the largest double
// below 1, as libstdc++ does.
__device__ __forceinline__ double canonical53(uint32_t w1, uint32_t w2)
{
    double sum = 0.0;
    sum += (double)w1 * 1.0;
    sum += (double)w2 * 4294967296.0;
    double r = sum / 18446744073709551616.0;
    if (r >= 1.0) r = 0x1.fffffffffffffp-1; // nextafter(1, 0)
    return r;
}

} // namespace ompl_amd
