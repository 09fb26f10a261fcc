// Device helpers of the batched check kernels: reading configurations, the
// outcome of an edge's s2 check, and the survivor list.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>

#include "checker.hpp"
#include "motion_device.hpp"
#include "walk_device.hpp"

namespace ompl_amd {

// Configuration i of a dof-major array (n entries per joint) as FP32, zeros
// for a dead lane, which reads entry `fallback` (a valid index) and drops it:
// unconditional reads are issued together and wait for one memory round trip,
// where reads under the lane's condition were issued and awaited a few at a time.
template <typename T>
__device__ __forceinline__ void load_config(const T *soa, int64_t n, int64_t i, bool live, float q[kDof],
                                            int64_t fallback = 0)
{
    const int64_t ic = live ? i : fallback;
    T v[kDof];
#pragma unroll
    for (int j = 0; j < kDof; ++j) v[j] = soa[(int64_t)j * n + ic];
#pragma unroll
    for (int j = 0; j < kDof; ++j) q[j] = live ? (float)v[j] : 0.0f;
}

// Result of an edge's s2 check (H: folded hit mask of the wave) on the group
// leader: writes the final result of every edge that needs no walk and
// returns true for a survivor (s2 valid, 2 <= nd <= kMaxSegments), m = nd - 1.
template <int GS>
__device__ __forceinline__ bool endpoint_finish(const MotionArgs &A, int64_t e, bool live, uint64_t H, int &m,
                                                double a[kDof], double b[kDof])
{
    const int lane = lane_id();
    m = 0;
    if (!live || lane % GS != 0) return false;
    const bool s2_valid = !((H >> lane) & 1);
    if (!s2_valid) {
        A.out[e] = 0;
        if (A.checked) A.checked[e] = 1;
        return false;
    }
#pragma unroll
    for (int j = 0; j < kDof; ++j) {
        a[j] = A.a[(int64_t)j * A.n + e];
        b[j] = A.b[(int64_t)j * A.n + e];
    }
    const int nd = valid_segment_count<kDof>(a, b, A.lvs, A.factor);
    if (nd > kMaxSegments) {
        A.out[e] = 0;
        if (A.checked) A.checked[e] = 0;
        return false;
    }
    if (nd < 2) {
        A.out[e] = 1;
        if (A.checked) A.checked[e] = 1;
        return false;
    }
    m = nd - 1;
    return true;
}

// Block-aggregated append of the survivors to the list, with their segment
// count and endpoints.  Every thread of the block calls it (it holds three
// barriers); a survivor's slot is returned.  The waves' counts meet in LDS, and
// one thread per block makes the device-wide atomic: device-scope atomics on one
// address from every CU serialise, and with many survivors (a sparse scene) one
// atomic per survivor cost more than the s2 checks themselves.
__device__ __forceinline__ int append_survivor(const MotionArgs &A, int64_t e, bool survivor, int m,
                                               const double a[kDof], const double b[kDof])
{
    __shared__ int blk_count, blk_base;
    const int lane = lane_id();
    if (threadIdx.x == 0) blk_count = 0;
    __syncthreads();
    const uint64_t sm = wave_ballot(survivor);
    int woff = 0;
    if (sm) {
        if (lane == lowest_bit(sm)) woff = atomicAdd(&blk_count, __popcll(sm));
        woff = __shfl(woff, lowest_bit(sm));
    }
    __syncthreads();
    if (threadIdx.x == 0 && blk_count > 0) blk_base = atomicAdd(A.list_count, blk_count);
    __syncthreads();
    const int slot = blk_base + woff + __popcll(sm & (((uint64_t)1 << lane) - 1));
    if (survivor) {
        A.out[e] = 1; // until the walk finds an invalid position
        A.list[slot] = (int32_t)e;
        A.surv_nd[slot] = m + 1;
        double *ab = A.surv_ab + (int64_t)slot * 2 * kDof;
#pragma unroll
        for (int j = 0; j < kDof; ++j) {
            ab[j] = a[j];
            ab[kDof + j] = b[j];
        }
    }
    return slot;
}

} // namespace ompl_amd
