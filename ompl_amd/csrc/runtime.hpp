// Runtime state shared by the C-ABI translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <atomic>
#include <mutex>
#include <vector>

#include "checker.hpp"
#include "common.hpp"

namespace ompl_amd {

void init_device(int dev);
// Takes the device address of the no-allocation entry point's scratch array
// (once per device, with that device current).
void init_noalloc_scratch(int dev);

// Device memory of objects that come and go (roadmaps, nearest-neighbour
// structures): a block given back is kept for the next taker, up to
// kKeptBlocksBytes in all, and kept blocks go back to the device when an
// allocation of the library fails (device_malloc).  The giver sees to it that nothing on the device still
// uses the block.  Safe from any thread.
struct DeviceBlock {
    void *p = nullptr;
    size_t bytes = 0;
};
constexpr size_t kKeptBlocksBytes = (size_t)768 << 20;
DeviceBlock take_block(size_t bytes);
void give_block(const DeviceBlock &b);
// hipMalloc and hipMallocAsync; when the device is out of memory the kept blocks
// go back to it and the allocation is tried again.
hipError_t device_malloc_bytes(void **p, size_t bytes);
hipError_t device_malloc_async_bytes(void **p, size_t bytes, hipStream_t s);
template <class T>
hipError_t device_malloc(T **p, size_t bytes)
{
    return device_malloc_bytes(reinterpret_cast<void **>(p), bytes);
}
template <class T>
hipError_t device_malloc_async(T **p, size_t bytes, hipStream_t s)
{
    return device_malloc_async_bytes(reinterpret_cast<void **>(p), bytes, s);
}

// Per-stream scratch of the batched motion path: survivor list + counters.
struct Workspace {
    int32_t *list = nullptr;    // survivors' edges
    int32_t *surv_nd = nullptr; // their segment counts
    double *surv_ab = nullptr;  // and endpoints a, b (14 doubles)
    int32_t *rest = nullptr;    // whether an item is unfinished
    int32_t *longs = nullptr;   // three words per entry: long items
    size_t list_cap = 0;
    // two sets of two at [16..17] and [20..21] (apart from each other's cache
    // sector), used in turn by grid_parity, each cleared by the batch before;
    // a third at [32..33] for batches that a caller captures (and [36..37], which
    // they clear in place of the next batch's); from [64] on a word and a ticket
    // per item of a one-launch batch
    int32_t *counters = nullptr;
    int grid_parity = 0;
    bool captured = false; // a caller's graph uses the arrays: outgrown, they stay allocated
    // Held by a batch from choosing its counter set to enqueuing its launches
    // (and around resizing), so host threads that share a stream cannot pick
    // the same set or see arrays being replaced.
    std::mutex mu;
};
// The stream's workspace with room for list_entries survivors.  The caller
// must hold the returned workspace's mu while it uses the workspace (lock
// passes that lock back, already taken, before any resize).
// Arrays of a workspace for `cap` survivors (counters excepted); freed with free_workspace_arrays.
void alloc_workspace_arrays(Workspace &w, size_t cap);
void free_workspace_arrays(Workspace &w);
// The next grid batch's view of a workspace (its lock held).
GridScratch grid_scratch(Workspace &w);
// The same of stream s's workspace.  While the caller captures s the batch gets
// the set for captured batches and a launch that clears it: each replay then
// starts from zero counts, whatever ran between, and leaves the other sets alone.
GridScratch stream_grid_scratch(Workspace &w, hipStream_t s);
Workspace &workspace(hipStream_t s, size_t list_entries, std::unique_lock<std::mutex> &lock);

// Per-thread stream and pinned result slot of the blocking single-call entry
// points (OMPL checkers must be thread-safe: base/StateValidityChecker.h:87-89).
struct ThreadResources {
    hipStream_t stream = nullptr;
    int32_t *pinned = nullptr;     // 4 KiB, host-coherent, device-mapped
    int32_t *pinned_dev = nullptr; // device address of the same memory
    char *stage = nullptr;         // growable host-coherent, device-mapped staging
    char *stage_dev = nullptr;
    size_t stage_cap = 0;
};
ThreadResources &thread_resources();
// Ensures r.stage holds `bytes` (callers synchronize r.stream before reuse).
void stage_reserve(ThreadResources &r, size_t bytes);

// Launch shapes (mirrors ompl_amd_tuning).
struct Tuning {
    int validity_lanes_per_state;
    int validity_obstacle_parts;
    int validity_block;
    int motion_lanes_per_state;
    int motion_obstacle_parts;
    int motion_block;
    int motion_waves_per_cu;
    int motion_strategy;
    int validity_shared_fk = 0;
};

Tuning get_tuning();
// Rejects (OA_REQUIRE) a tuning whose shapes or limits are not built.
void check_tuning(const Tuning &t);

struct Env;
// Batched DiscreteMotionValidator::checkMotion(s1, s2) over device arrays with
// launch shapes t; `own` supplies the survivor workspace (null: the stream's).
void check_motions_tuned(const Tuning &t, const Env &env, const double *a, const double *b, int64_t n, double lvs,
                         unsigned factor, uint8_t *out, int32_t *checked, hipStream_t s, Workspace *own = nullptr);
void set_tuning(const Tuning &t);
ompl_amd_tuning tuning_to_c(const Tuning &x);
Tuning tuning_from_c(const ompl_amd_tuning &t);

// Device-resident obstacle set.
struct Env {
    // ns spheres (x,y,z,(R+r)^2), then nb boxes as (lo),(hi), in the caller's
    // order, for the reference-order work accounting only
    float4 *obs = nullptr;
    GridView grid{}; // cell grid (grid.hpp), in the same allocation
    int ns = 0;
    int nb = 0;
    size_t bytes = 0;
    EnvView view() const { return EnvView{obs, ns, nb}; }
};

// A planning query on a batch PRM roadmap (prm.hip): start and goal become
// milestones 0 and 1 of a roadmap over n_samples uniform samples (n_streams
// generators seeded seed, seed + 1, ...) with k neighbours per milestone; the
// path is the shortest one between them over the valid edges.
struct PrmQuery {
    bool solved = false;
    int64_t milestones = 0, candidate_edges = 0, valid_edges = 0;
    std::vector<double> path; // row-major states
};
PrmQuery prm_query(ompl_amd_env env, const double start[7], const double goal[7], uint32_t seed, int n_streams,
                   int64_t n_samples, int k, double lvs, unsigned factor, hipStream_t s);
// Device bytes a prm_query of n_samples with k neighbours may hold at once (an upper estimate).
size_t prm_footprint(int64_t n_samples, int k);
// Shortest path between milestones 0 and 1 of a symmetric CSR roadmap.
std::vector<int32_t> roadmap_shortest_path(const std::vector<int64_t> &off, const std::vector<int32_t> &adj,
                                           const std::vector<double> &nodes);

// Largest obstacle set of an environment (float4 words).
constexpr int kMaxEnvWords = 4096;

} // namespace ompl_amd

struct ompl_amd_env_s {
    ompl_amd::Env env;
    // server requests (queued or running) that read this environment;
    // ompl_amd_env_destroy refuses while any remain
    std::atomic<int> server_users{0};
    // launch shapes of this environment's batched checks, when set; else the
    // library's current tuning
    mutable std::mutex tuning_mutex;
    bool has_tuning = false;
    ompl_amd::Tuning tuning{};
};

namespace ompl_amd {
// The tuning the batched checks on environment e use.
Tuning tuning_for(const ompl_amd_env_s &e);
} // namespace ompl_amd
