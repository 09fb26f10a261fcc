// Launch shapes a tuning may name, clearing of counters, and the arm's sphere
// centres.  The checks themselves are in grid_check.hip.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "arm_device.hpp"
#include "checker.hpp"

namespace ompl_amd {

bool shape_supported(int lps, int ops)
{
    return (ops == 1 && (lps == 1 || lps == 2 || lps == 4 || lps == 7 || lps == 8)) ||
           (lps == 8 && (ops == 2 || ops == 4 || ops == 8)) || (lps == 7 && (ops == 2 || ops == 4 || ops == 9));
}

bool fused_supported(int le, int oe, int lw, int ow)
{
    const bool e_ok = le == 8 && (oe == 1 || oe == 2 || oe == 4);
    const bool w_ok = (lw == 1 && ow == 1) || (lw == 8 && (ow == 1 || ow == 8));
    return e_ok && w_ok;
}

__global__ void zero_ints_kernel(int *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void arm_spheres_kernel(const float *__restrict__ q_soa, int64_t n, float *__restrict__ out)
{
    const int64_t st = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (st >= n) return;
    float q[kDof];
#pragma unroll
    for (int j = 0; j < kDof; ++j) q[j] = q_soa[(int64_t)j * n + st];
    ArmSpheres S;
    arm_fk(q, S);
#pragma unroll
    for (int m = 0; m < kSpheres; ++m) {
        out[(st * kSpheres + m) * 3 + 0] = S.x[m];
        out[(st * kSpheres + m) * 3 + 1] = S.y[m];
        out[(st * kSpheres + m) * 3 + 2] = S.z[m];
    }
}

void launch_zero(int *p, int n, hipStream_t s)
{
    hipLaunchKernelGGL(zero_ints_kernel, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    OA_HIP(hipGetLastError());
}

void launch_arm_spheres(const float *q, int64_t n, float *out, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(arm_spheres_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, q, n, out);
    OA_HIP(hipGetLastError());
}

} // namespace ompl_amd
