// Device-side arm model: FP32 forward kinematics of the 7-DOF sphere arm and
// the sphere/sphere, sphere/box collision predicates.  Operation order (fixed;
// -ffp-contract=off):
//
//   joint i (axis z for even i, y for odd i), (s, c) = sincos_pl(q_i):
//     z joint: X' = X*c + Y*s,  Y' = Y*c - X*s   (per component)
//     y joint: X' = X*c - Z*s,  Z' = X*s + Z*c
//   sphere j of link i: centre = p_i + Z_i * off_j, off = {0.0375, 0.1125,
//     0.1875, 0.2625} (link 0.3 m, fractions 1/8, 3/8, 5/8, 7/8), r = 0.05
//   p_{i+1} = p_i + Z_i * 0.3
//   sphere obstacle (o, R): d = o - centre, d2 = (dx*dx + dy*dy) + dz*dz,
//     collision iff d2 < rr, rr = (R + 0.05f) * (R + 0.05f)
//   box obstacle (lo = b - h, hi = b + h): p = min(max(centre, lo), hi),
//     d = centre - p, d2 = (dx*dx + dy*dy) + dz*dz, collision iff d2 < 0.05f*0.05f
//
// The reference's own FP32 checker (VAMP, vamp/VampStateValidityChecker.h:37-41)
// is an absent submodule; this arm and these predicates are the project's
// specification of the checker behind StateValidityChecker::isValid.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fp32_math.hpp"

namespace ompl_amd {

constexpr int kDof = 7;
constexpr int kSpheres = 28;
constexpr float kLink = 0.3f;
constexpr float kRobotR = 0.05f;

__device__ __forceinline__ float sphere_offset(int j)
{
    return j == 0 ? 0.0375f : (j == 1 ? 0.1125f : (j == 2 ? 0.1875f : 0.2625f));
}

// Obstacles: [0, ns) spheres (x, y, z, rr); then nb boxes as pairs (lo.xyz,
// 0), (hi.xyz, 0).
struct EnvView {
    const float4 *obs;
    int ns;
    int nb;
};

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own
// L2.  This permutation gives XCD x a contiguous run of logical blocks
// (hardware block b = 8 i + x -> the i-th block of XCD x's run; the first
// nb % 8 XCDs get one block more), so that neighbouring states, which share
// cache lines of the dof-major arrays, are fetched into one L2 only.
__device__ __forceinline__ int64_t xcd_block(int64_t b, int64_t nb)
{
    const int64_t q = nb >> 3, r = nb & 7, x = b & 7, i = b >> 3;
    return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + i;
}

// The sphere centres of one state.
struct ArmSpheres {
    float x[kSpheres], y[kSpheres], z[kSpheres];
};

// Frame (P, W) of link g from the sines and cosines that lanes 0 .. 6 of the
// state's GS lanes hold, one joint each; the rotation chain is the one arm_fk
// evaluates.
template <int GS>
__device__ __forceinline__ void link_chain(float sm, float cm, int g, float P[3], float W[3])
{
    float sj[kDof], cj[kDof];
#pragma unroll
    for (int i = 0; i < kDof; ++i) {
        const int src = (threadIdx.x & 63 & ~(GS - 1)) + i;
        sj[i] = __shfl(sm, src);
        cj[i] = __shfl(cm, src);
    }
    float X0 = 1.0f, X1 = 0.0f, X2 = 0.0f;
    float Y0 = 0.0f, Y1 = 1.0f, Y2 = 0.0f;
    float Z0 = 0.0f, Z1 = 0.0f, Z2 = 1.0f;
    float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f;
    float P0 = 0.0f, P1 = 0.0f, P2 = 0.0f, W0 = 0.0f, W1 = 0.0f, W2 = 1.0f;
#pragma unroll
    for (int i = 0; i < kDof; ++i) {
        const float s = sj[i], c = cj[i];
        if ((i & 1) == 0) {
            float nx0 = X0 * c + Y0 * s, ny0 = Y0 * c - X0 * s;
            float nx1 = X1 * c + Y1 * s, ny1 = Y1 * c - X1 * s;
            float nx2 = X2 * c + Y2 * s, ny2 = Y2 * c - X2 * s;
            X0 = nx0; X1 = nx1; X2 = nx2;
            Y0 = ny0; Y1 = ny1; Y2 = ny2;
        } else {
            float nx0 = X0 * c - Z0 * s, nz0 = X0 * s + Z0 * c;
            float nx1 = X1 * c - Z1 * s, nz1 = X1 * s + Z1 * c;
            float nx2 = X2 * c - Z2 * s, nz2 = X2 * s + Z2 * c;
            X0 = nx0; X1 = nx1; X2 = nx2;
            Z0 = nz0; Z1 = nz1; Z2 = nz2;
        }
        const bool mine = g == i;
        P0 = mine ? p0 : P0;
        P1 = mine ? p1 : P1;
        P2 = mine ? p2 : P2;
        W0 = mine ? Z0 : W0;
        W1 = mine ? Z1 : W1;
        W2 = mine ? Z2 : W2;
        p0 = p0 + Z0 * kLink;
        p1 = p1 + Z1 * kLink;
        p2 = p2 + Z2 * kLink;
    }
    P[0] = P0;
    P[1] = P1;
    P[2] = P2;
    W[0] = W0;
    W[1] = W1;
    W[2] = W2;
}

// All sphere centres by one lane.
__device__ __forceinline__ void arm_fk(const float q[kDof], ArmSpheres &S)
{
    float X0 = 1.0f, X1 = 0.0f, X2 = 0.0f;
    float Y0 = 0.0f, Y1 = 1.0f, Y2 = 0.0f;
    float Z0 = 0.0f, Z1 = 0.0f, Z2 = 1.0f;
    float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f;
#pragma unroll
    for (int i = 0; i < kDof; ++i) {
        float s, c;
        sincos_pl(q[i], s, c);
        if ((i & 1) == 0) {
            float nx0 = X0 * c + Y0 * s, ny0 = Y0 * c - X0 * s;
            float nx1 = X1 * c + Y1 * s, ny1 = Y1 * c - X1 * s;
            float nx2 = X2 * c + Y2 * s, ny2 = Y2 * c - X2 * s;
            X0 = nx0; X1 = nx1; X2 = nx2;
            Y0 = ny0; Y1 = ny1; Y2 = ny2;
        } else {
            float nx0 = X0 * c - Z0 * s, nz0 = X0 * s + Z0 * c;
            float nx1 = X1 * c - Z1 * s, nz1 = X1 * s + Z1 * c;
            float nx2 = X2 * c - Z2 * s, nz2 = X2 * s + Z2 * c;
            X0 = nx0; X1 = nx1; X2 = nx2;
            Z0 = nz0; Z1 = nz1; Z2 = nz2;
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const float off = sphere_offset(m);
            S.x[4 * i + m] = p0 + Z0 * off;
            S.y[4 * i + m] = p1 + Z1 * off;
            S.z[4 * i + m] = p2 + Z2 * off;
        }
        p0 = p0 + Z0 * kLink;
        p1 = p1 + Z1 * kLink;
        p2 = p2 + Z2 * kLink;
    }
}

// min(max(x, lo), hi) for finite lo <= hi (every stored box: coordinates are
// checked finite and extents non-negative when an environment is created) in
// one instruction: v_med3_f32 returns the same bits as the min/max pair for
// every x (a NaN x gives a NaN distance either way), without the
// canonicalising moves IEEE-mode min/max need.
__device__ __forceinline__ float clamp_box(float x, float lo, float hi)
{
    return __builtin_amdgcn_fmed3f(x, lo, hi);
}

// Wave-level helpers (wave64).
__device__ __forceinline__ uint64_t wave_ballot(bool p)
{
    return __ballot(p);
}

// Bits set at the first lane of every LPS-lane group.
template <int LPS>
__host__ __device__ constexpr uint64_t leader_mask()
{
    uint64_t m = 0;
    for (int i = 0; i < 64; i += LPS) m |= (uint64_t)1 << i;
    return m;
}

// Folds a per-lane mask onto group leaders: bit (g*LPS) set iff any lane of
// group g is set.
template <int LPS>
__device__ __forceinline__ uint64_t fold_groups(uint64_t m)
{
#pragma unroll
    for (int sh = 1; sh < LPS; sh <<= 1) m |= m >> sh;
    return m & leader_mask<LPS>();
}

} // namespace ompl_amd
