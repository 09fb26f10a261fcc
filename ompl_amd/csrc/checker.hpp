// Host-visible argument blocks and launchers of the checker kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "arm_device.hpp"
#include "common.hpp"
#include "grid.hpp"

namespace ompl_amd {

struct MotionArgs {
    const double *a; // FP64 [7][n] dof-major
    const double *b;
    int64_t n;
    double lvs;
    unsigned factor;
    uint8_t *out;
    int32_t *checked;    // optional
    int32_t *list;       // survivors of the s2 pass: their edges,
    int32_t *list_count; // number,
    int32_t *surv_nd;    // segment counts
    double *surv_ab;     // and endpoints, a then b (14 doubles)
};

struct Edge1 {
    double a[kDof];
    double b[kDof];
};

struct State1 {
    double q[kDof];
};

// Launch shapes and one-launch shape pairs a tuning may name.
bool shape_supported(int lps, int ops);
bool fused_supported(int le, int oe, int lw, int ow);
void launch_zero(int *p, int n, hipStream_t s);
// Edges or lists up to which a block each walks them in one launch: 1,024
// blocks of four waves are one wave per SIMD, so the speculative positions of
// edges that fail at once cost no time; more edges go through the s2 pass.
constexpr int kWideItems = 1024;
// Ints of a workspace's counters, zero at its creation.
constexpr int kWorkspaceCounters = 64 + 2 * kWideItems;
// Survivor workspace of the checks over the cell grid (grid_check.hip).
struct GridScratch {
    int32_t *list, *surv_nd, *rest, *long_slot, *long_bad, *ticket; // an entry per edge or list
    double *surv_ab;                                                 // 14 per edge
    int32_t *wide;                                                   // 2 kWideItems words, zero between batches
    int32_t *counts;                                                 // two words, zero
    int32_t *next;                                                   // two words, cleared for the next batch
};
template <typename T>
void launch_grid_validate(const GridView &g, const T *q, int64_t n, uint8_t *out, hipStream_t s);
// fused: timed as one launch ("motion_fused") rather than by kernel.
void launch_grid_motions(const GridView &g, const MotionArgs &m, const GridScratch &w, bool fused, hipStream_t s);
// One edge or state, passed by value; *result: 1 valid, 0 not.
void launch_motion_single(const GridView &g, const Edge1 &E, double lvs, unsigned factor, int *result,
                          hipStream_t s);
void launch_validate_single(const GridView &g, const State1 &st, int *result, hipStream_t s);
void launch_grid_last_valid(const GridView &g, const MotionArgs &m, double *last_t, const GridScratch &w,
                            hipStream_t s);
void launch_grid_state_lists(const GridView &g, const double *q_soa, int64_t n_states, const int64_t *offsets,
                             int64_t n_lists, uint8_t *out, int32_t *first_invalid, const GridScratch &w,
                             hipStream_t s);
void launch_arm_spheres(const float *q, int64_t n, float *out, hipStream_t s);

} // namespace ompl_amd
