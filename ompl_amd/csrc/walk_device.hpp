// Device helpers shared by the batched motion kernels and the planning
// server: wave utilities and the walk of one edge in DiscreteMotionValidator
// order (position 0 = s2, positions p >= 1 = the p-th bisection check,
// base/src/DiscreteMotionValidator.cpp:93-145).
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "arm_device.hpp"
#include "motion_device.hpp"

namespace ompl_amd {

__device__ __forceinline__ int lane_id()
{
    return threadIdx.x & 63;
}

__device__ __forceinline__ int lowest_bit(uint64_t m)
{
    return __builtin_ctzll(m);
}

// State of walk position p (0 = b, else bisection index p-1) as FP32.
__device__ __forceinline__ void walk_state(const double a[kDof], const double b[kDof], int nd, int p, float q[kDof])
{
    if (p == 0) {
#pragma unroll
        for (int j = 0; j < kDof; ++j) q[j] = (float)b[j];
    } else {
        const int idx = bisection_index(p - 1, nd);
        interpolate_f32<kDof>(a, b, (double)idx / (double)nd, q);
    }
}

} // namespace ompl_amd
