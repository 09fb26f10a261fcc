// Exact distances of the nearest-neighbour searches, in the operation order
// of the CPU oracle (element minus query), and their sort keys.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fp32_math.hpp"
#include "../../include/ompl_amd.h"

namespace ompl_amd {

template <int METRIC, int DIM>
__device__ __forceinline__ float exact_dist(const float *__restrict__ e, const float q[DIM])
{
    if (METRIC == OMPL_AMD_METRIC_L2) {
        float dist = 0.0f;
#pragma unroll
        for (int i = 0; i < DIM; ++i) {
            const float diff = e[i] - q[i];
            dist += diff * diff;
        }
        return __builtin_sqrtf(dist);
    } else {
        float t = 0.0f;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const float diff = e[i] - q[i];
            t += diff * diff;
        }
        const float dt = __builtin_sqrtf(t);
        const float dq = fabsf(((e[3] * q[3] + e[4] * q[4]) + e[5] * q[5]) + e[6] * q[6]);
        const float dr = dq > 1.0f ? 0.0f : acos_as(dq);
        float dist = 0.0f;
        dist += 1.0f * dt;
        dist += 1.0f * dr;
        return dist;
    }
}

// SE3: true when the point's distance is certainly above `bound` (a finite
// distance), from a lower bound that skips the acos: acos(x) >= sqrt(2 (1 - x))
// on [0, 1] (2 sin(t / 2) <= t), so d >= d_t + sqrt(2 (1 - |q.x|)).  The margin
// (relative 1e-5 plus 1e-5) covers the FP32 rounding of both sides and
// acos_as's error, so a point this skips is one whose exact distance is above
// the bound.  Other metrics: never.
template <int METRIC, int DIM>
__device__ __forceinline__ bool certainly_above(const float *__restrict__ e, const float q[DIM], float bound)
{
    if (METRIC != OMPL_AMD_METRIC_SE3) return false;
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float diff = e[i] - q[i];
        t += diff * diff;
    }
    const float dq = fabsf(((e[3] * q[3] + e[4] * q[4]) + e[5] * q[5]) + e[6] * q[6]);
    const float lb = __builtin_amdgcn_sqrtf(t) + __builtin_amdgcn_sqrtf(2.0f * (1.0f - dq));
    return lb > bound * (1.0f + 1e-5f) + 1e-5f; // false for NaN (dq > 1) or an infinite bound
}

__device__ __forceinline__ unsigned long long pack_key(float d, int i)
{
    return ((unsigned long long)__float_as_uint(d) << 32) | (uint32_t)i;
}

} // namespace ompl_amd
