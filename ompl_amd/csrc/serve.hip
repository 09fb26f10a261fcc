// Planning server: continuous batching of RRT-Connect requests on one GPU,
// each request's planner loop resident on the device.
//
// A request is a single-query RRT-Connect plan (geometric/planners/rrt/src/
// RRTConnect.cpp:116-196 growTree, :245-330 solve) on the 7-DOF arm in one of
// the registered environments, from one or more start states to one or more
// goal states (PlannerInputStates order, base/src/Planner.cpp:228-336).
// Everything the loop touches lives in one region of a device pool sized to
// the HBM budget: both trees (append-only FP64 states + parent indices), the
// start and goal states, the state sampler's mt19937 and the solve loop's
// variables, and the solution path.  The server thread launches slices: one
// block (512 threads, or 1,024) per active request runs its loop
// -- sample, nearest neighbour, steer, motion check, append, connect loop,
// path splice -- for a bounded time, then stores its state; the host then
// retires finished requests and admits queued ones while their region fits
// the pool (continuous batching), and launches the next slice.  A slice
// resumes each loop exactly where the last one stopped, so a request's result
// does not depend on the slices it ran in or the requests it shared them
// with.
//
// Inside a block: the nearest neighbour is an FP64 scan of the tree (first
// strict minimum), its first nodes in LDS, reduced by (distance, index); states
// are checked over the environment's cell grid (grid_device.hpp), eight lanes
// each where few are wanted at once and one lane each for the rest of a long
// motion; the sampler's draws are made a generator block at a time.
//
// A request is one chain of steps, so it is bound by latency: what counts is
// how many steps share one pass of it.  Most sampling steps are trapped, and a
// trapped step changes nothing but the draws, so up to 32 of them run at once
// (16 lanes each), the first valid one is committed, and the pass costs about
// 9 us.  64 requests over eight scenes of up to 128 obstacles, 48,900 steps,
// the longest request 2,128 of them: 3.3 ms (11.3 before: eight at
// a time, each tested against every obstacle, and copies of commands, results, end states and
// paths around every slice, which the kernel now reads and writes in pinned memory).
//
// Plain counterpart: ompl_amd_plan_plain runs the same RRT-Connect on the host
// with host nearest neighbours and one GPU launch + synchronisation per
// isValid / checkMotion call.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <deque>
#include <map>
#include <mutex>
#include <random>
#include <thread>
#include <unordered_map>
#include <vector>

#include "grid_device.hpp"
#include "mt_device.hpp"
#include "runtime.hpp"
#include "walk_device.hpp"

namespace ompl_amd {

enum GrowStatus { kTrapped = 0, kAdvanced = 1, kReached = 2 };

constexpr double kPi = 3.141592653589793238462643383279502884;
constexpr double kEqualEps = 2.220446049250313080847e-16 * 2.0; // StateSpace::equalStates (RealVector)
// Largest environment a request may name, as the bytes of its obstacles in
// lists padded to kPlanPad (60 KiB: 2,880 spheres or 1,728 boxes).  The kernel no
// longer stages them; the limit is what callers know.
constexpr int kPlanPad = 288;
constexpr size_t kPlanMaxEnvBytes = 60 * 1024;
// Start / goal states a request may list (each).
constexpr int kMaxEnds = OMPL_AMD_MAX_ENDPOINTS;

// Persistent state of one request's RRTConnect::solve loop (device).
struct PlanState {
    uint32_t mt[kMtN]; // the state sampler's RNG (std::mt19937)
    int32_t mti;       // next word (kMtN: twist first)
    int32_t status;
    int32_t iteration;
    int32_t n0, n1;     // nodes of the start / goal tree
    int32_t start_tree; // RRTConnect::startTree_
    int32_t tgi_start;  // tgi.start
    int32_t grow_tree;  // tree of the next growTree (0 start, 1 goal)
    int32_t phase;      // 0: sample + grow, 1: first connect step, 2: connect loop
    int32_t added, xmotion;
    int32_t path_len;
    int32_t sampled_goals; // goal states handed out so far (PlannerInputStates)
    int64_t steps, checks;
    double rstate[kDof];
};

__host__ __device__ inline size_t align256(size_t b)
{
    return (b + 255) & ~(size_t)255;
}

// One request's region: [start tree states][goal tree states][start parents]
// [goal parents][path states][path node indices][start and goal states]
// [PlanState].  Tree states
// are dof-major (coordinate k of node i at k * cap + i), so a wave's reads of
// consecutive nodes coalesce; the path is row-major.
struct RegionPtrs {
    double *tree_s[2];
    int32_t *parent[2];
    double *path;
    int32_t *path_idx;
    double *ends; // kMaxEnds start rows, then kMaxEnds goal rows
    PlanState *state;
    size_t bytes;
};

__host__ __device__ inline RegionPtrs region_ptrs(char *base, int cap)
{
    RegionPtrs R;
    size_t off = 0;
    for (int t = 0; t < 2; ++t) {
        R.tree_s[t] = reinterpret_cast<double *>(base + off);
        off += align256((size_t)cap * kDof * sizeof(double));
    }
    for (int t = 0; t < 2; ++t) {
        R.parent[t] = reinterpret_cast<int32_t *>(base + off);
        off += align256((size_t)cap * sizeof(int32_t));
    }
    R.path = reinterpret_cast<double *>(base + off);
    off += align256((size_t)2 * cap * kDof * sizeof(double));
    R.path_idx = reinterpret_cast<int32_t *>(base + off);
    off += align256((size_t)2 * cap * sizeof(int32_t));
    R.ends = reinterpret_cast<double *>(base + off);
    off += align256((size_t)2 * kMaxEnds * kDof * sizeof(double));
    R.state = reinterpret_cast<PlanState *>(base + off);
    off += align256(sizeof(PlanState));
    R.bytes = off;
    return R;
}

static size_t footprint(int max_nodes)
{
    return region_ptrs(nullptr, max_nodes).bytes;
}

// Per active request and slice (a host array that the kernel reads once).
struct PlanCmd {
    GridView grid; // the environment
    char *region;
    int32_t cap;       // nodes per tree
    int32_t max_iters;
    double maxd;       // maxDistance_
    double lvs;        // longest valid segment
    uint32_t factor;
    uint32_t seed;
    int32_t init;      // 1: first slice (seed the sampler, plant the roots)
    int32_t n_starts, n_goals; // rows of the region's start and goal states
    int32_t inter;     // addIntermediateStates
    const double *ends; // first slice: the start and goal rows, as in the region (host memory)
    double *path;       // where a solution of at most SliceArgs::path_rows rows goes (host memory), else the region
};

// Per active request, written at the end of each slice.  t_*: device
// wall-clock ticks this slice spent sampling, in nearest-neighbour scans, in
// motion checks (steering included) and in whole growTree steps.
struct PlanOut {
    int32_t status, iteration, n0, n1, path_len, pad;
    int64_t steps, checks;
    int64_t t_sample, t_nearest, t_check, t_step;
};

// Longest solution written to pinned memory by the slice that finds it (a longer
// one is copied from its region), within kPathBytes for all active requests.
constexpr int kPathRows = 128;
constexpr size_t kPathBytes = (size_t)16 << 20;

struct SliceArgs {
    const PlanCmd *cmds; // host memory, as is out: read and written once, no copies around a slice
    PlanOut *out;
    int path_rows;
    int64_t budget; // wall-clock ticks per slice (at least one step is always made)
};

static size_t env_stage_bytes(int ns, int nb)
{
    auto pad = [](int n) { return (n + kPlanPad - 1) / kPlanPad * kPlanPad; };
    return (size_t)(pad(ns) + 2 * pad(nb)) * sizeof(float4) + (size_t)ns * sizeof(float);
}

// Candidate nearest node: its distance and index; the lower index wins a tie.
struct Near {
    double d = INFINITY;
    int i = INT_MAX;
    __device__ __forceinline__ void take(double od, int oi)
    {
        if (od < d || (od == d && oi < i)) {
            d = od;
            i = oi;
        }
    }
    template <int CTRL>
    __device__ __forceinline__ void dpp()
    {
        const long long u = __double_as_longlong(d);
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, 0xf, 0xf, true);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, 0xf, 0xf, true);
        const int oi = __builtin_amdgcn_update_dpp(0, i, CTRL, 0xf, 0xf, true);
        take(__longlong_as_double((long long)(((unsigned long long)hi << 32) | lo)), oi);
    }
    // The best of each group of `lanes` (16 or 64) in all its lanes.
    __device__ __forceinline__ void share(int lanes)
    {
        dpp<0x128>(); // row_ror 8, 4, 2, 1: rows of 16 lanes
        dpp<0x124>();
        dpp<0x122>();
        dpp<0x121>();
        if (lanes == 64) {
            take(__shfl_xor(d, 16), __shfl_xor(i, 16));
            take(__shfl_xor(d, 32), __shfl_xor(i, 32));
        }
    }
};

constexpr int kKeptNodes = 256; // of each tree, in LDS

// A tree: its nodes (dof-major with stride cap), the first `kept` of them also
// in LDS (stride kept).
struct Tree {
    double *T, *lds;
    int cap;
    static constexpr int kept = kKeptNodes;
    __device__ __forceinline__ double at(int k, int i) const
    {
        return i < kept ? lds[k * kept + i] : T[(int64_t)k * cap + i];
    }
    __device__ __forceinline__ void set(int k, int i, double v) const
    {
        T[(int64_t)k * cap + i] = v;
        if (i < kept) lds[k * kept + i] = v;
    }
};

// Nearest of n nodes to tgt among nodes first, first + stride, ..: first strict
// minimum of distance(node, tgt) (NearestNeighborsLinear::nearest order).
__device__ __forceinline__ Near scan_nearest(const Tree &t, int n, const double tgt[kDof], int first, int stride)
{
    Near best;
    double best2 = INFINITY; // a squared distance no smaller has no smaller root
    auto distance2 = [&](int i, const double *T, int64_t step) {
        double dist = 0.0;
#pragma unroll
        for (int k = 0; k < kDof; ++k) {
            const double diff = T[k * step + i] - tgt[k];
            dist += diff * diff;
        }
        return dist;
    };
    auto take = [&](int i, double dist) {
        if (dist < best2) {
            const double d = __builtin_sqrt(dist);
            best2 = dist;
            if (d < best.d) { // indices increase: strict < keeps the lowest
                best.d = d;
                best.i = i;
            }
        }
    };
    int i = first;
    for (; i < min(n, t.kept); i += stride) take(i, distance2(i, t.lds, t.kept));
    constexpr int kAtOnce = 4; // nodes whose reads are in flight together
    for (; i < n; i += kAtOnce * stride) {
        double d2[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) d2[u] = distance2(min(i + u * stride, n - 1), t.T, t.cap);
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u)
            if (i + u * stride < n) take(i + u * stride, d2[u]);
    }
    return best;
}

// The same over the whole tree by the whole block; every thread returns it.
template <int NT>
__device__ __forceinline__ Near block_nearest(const Tree &t, int n, const double tgt[kDof], double *s_wd, int *s_wi)
{
    Near best = scan_nearest(t, n, tgt, threadIdx.x, NT);
    best.share(64);
    if (lane_id() == 0) {
        s_wd[threadIdx.x >> 6] = best.d;
        s_wi[threadIdx.x >> 6] = best.i;
    }
    __syncthreads();
    best.d = s_wd[0];
    best.i = s_wi[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) best.take(s_wd[w], s_wi[w]);
    return best;
}

// growTree's new state (RRTConnect.cpp:116-135): the nearest node nst (made
// node 0 where no distance is finite), the target or, farther than maxd, the
// state maxd from nst towards it.
struct Steer {
    double nst[kDof], x[kDof];
    int nm;
    bool reach, moved; // not moved: no progress, TRAPPED without a check
    __device__ __forceinline__ void run(const Tree &t, int n, const Near &best, const double tgt[kDof], double maxd)
    {
        nm = best.i < n ? best.i : 0;
        double dd = best.d;
        double dist = 0.0;
#pragma unroll
        for (int k = 0; k < kDof; ++k) {
            nst[k] = t.at(k, nm);
            x[k] = tgt[k];
        }
        if (best.i >= n) {
#pragma unroll
            for (int k = 0; k < kDof; ++k) {
                const double diff = nst[k] - tgt[k];
                dist += diff * diff;
            }
            dd = __builtin_sqrt(dist);
        }
        reach = moved = true;
        if (dd > maxd) {
            const double s = maxd / dd;
            bool equal = true;
#pragma unroll
            for (int k = 0; k < kDof; ++k) {
                x[k] = nst[k] + (tgt[k] - nst[k]) * s;
                if (fabs(nst[k] - x[k]) > kEqualEps) equal = false;
            }
            moved = !equal;
            reach = false;
        }
    }
};

// A growTree step's motion: npos positions, the DiscreteMotionValidator's of
// (a, b) (0 = b, then the bisection order), or with `extra`, where b is a tree
// node, isValid(dst) first and b last.  a, b and dst are in LDS (read per
// round; no registers held across).  Validity of the whole motion does not
// depend on the order positions are visited in.
struct StepMotion {
    const double *a, *b, *dst;
    int nd, npos;
    bool extra;
    static __device__ __forceinline__ int positions(int nd, bool extra)
    {
        return 1 + (nd >= 2 ? nd - 1 : 0) + (extra ? 1 : 0);
    }
    // the state of position p if it is one of the motion's ends, else null
    __device__ __forceinline__ const double *end(int p) const
    {
        return !extra ? (p == 0 ? b : nullptr) : p == 0 ? dst : p == npos - 1 ? b : nullptr;
    }
    __device__ __forceinline__ double fraction(int p) const
    {
        return (double)bisection_index(p - 1, nd) / (double)nd;
    }
    // Eight lanes per position: joint j of position p.
    __device__ __forceinline__ float joint(int p, int j) const
    {
        if (const double *e = end(p)) return (float)e[j];
        const double t = fraction(p);
        return (float)(a[j] + (b[j] - a[j]) * t);
    }
    // One lane per position.
    __device__ __forceinline__ void state(int p, float q[kDof]) const
    {
        if (const double *e = end(p)) {
#pragma unroll
            for (int k = 0; k < kDof; ++k) q[k] = (float)e[k];
        } else {
            interpolate_f32<kDof>(a, b, fraction(p), q);
        }
    }
};

// Eight lanes per position: whether the lane finds position p (if there is
// one) invalid.
__device__ __forceinline__ bool wave_hit8(const GridView &g, const StepMotion &M, int p, WaveTests &tests)
{
    const bool live = p < M.npos;
    return state_hit8(g, M.joint(live ? p : 0, min(lane_id() & 7, kDof - 1)), live, tests);
}

// Positions from `first` on of a motion by the whole block, one lane each:
// false at the first round holding an invalid position.
template <int NT>
__device__ __forceinline__ bool block_check(const GridView &g, const StepMotion &M, int first, WaveTests *tests)
{
    for (int base = first; base < M.npos; base += NT) {
        const int p = base + (int)threadIdx.x;
        const bool live = p < M.npos;
        bool hit = false;
        if (wave_ballot(live)) {
            float q[kDof];
            M.state(live ? p : 0, q);
            hit = state_hit1(g, q, live, tests[threadIdx.x >> 6]);
        }
        if (__syncthreads_or(hit)) return false;
    }
    return true;
}

// SpaceInformation::satisfiesBounds && isValid of state q (global memory) by
// the whole block (PlannerInputStates, base/src/Planner.cpp:243-245): within
// machine epsilon of [-pi, pi] per joint (RealVectorStateSpace.cpp:200-208),
// then the checker.  q is staged in sx.
__device__ __forceinline__ bool endpoint_usable(const GridView &g, const double *q, double *sx, WaveTests *tests)
{
    if (threadIdx.x < kDof) sx[threadIdx.x] = q[threadIdx.x];
    __syncthreads();
    const double eps = 2.220446049250313080847e-16;
    bool in = true;
#pragma unroll
    for (int k = 0; k < kDof; ++k)
        if (sx[k] - eps > kPi || sx[k] + eps < -kPi) in = false;
    if (!in) return false; // block-uniform: every thread read the same state
    // every wave checks the one state
    const StepMotion M{sx, sx, sx, 0, 1, true};
    return wave_ballot(wave_hit8(g, M, lane_id() >> 3, tests[threadIdx.x >> 6])) == 0;
}

// Appends a valid growTree step to tree (t, P) after node nm: the new state x,
// or with addIntermediateStates (RRTConnect.cpp:148-183) the states of
// getMotionStates(a, b, validSegmentCount(a, b) = nd, endpoints) --
// a + (b - a) j / (nd + 1) -- without the tree's own end: from the start tree
// (a = nearest, b = x) states 1 .. nd + 1, from the goal tree (a = x, b =
// nearest) states nd .. 0, each the parent of the next.  Returns the index of
// the last (the new state), or -1 when the tree cannot hold them.
template <int NT>
__device__ int append_step(const Tree &t, int32_t *P, int &n, int nm, const double *a, const double *b,
                           const double *x, int nd, bool from_start, bool inter)
{
    const int tid = threadIdx.x;
    if (!inter) {
        if (n + 1 > t.cap) return -1;
        if (tid < kDof) t.set(tid, n, x[tid]);
        if (tid == 0) P[n] = nm;
        return n++;
    }
    const int seg = nd + 1;
    if (n + seg > t.cap) return -1;
    for (int i = tid; i < seg * kDof; i += NT) {
        const int r = i / kDof, k = i - r * kDof; // chain element r (0-based)
        const int j = from_start ? r + 1 : seg - 1 - r;
        double v;
        if (j == 0) v = a[k];
        else if (j == seg) v = b[k];
        else v = a[k] + (b[k] - a[k]) * ((double)j / (double)seg);
        t.set(k, n + r, v);
    }
    for (int r = tid; r < seg; r += NT) P[n + r] = r == 0 ? nm : n + r - 1;
    n += seg;
    return n - 1;
}

// Lanes of a speculative step, by the larger tree's size; it checks a position
// (the new state or s2 and what follows) with eight lanes each; those still
// open after them get a few more from whole waves, and the first that is then
// open is finished by the whole block.  While the nodes are in LDS a step costs
// the same in 16 lanes as in 64, and four times as many run at once; of a large
// tree's scan, the steps behind the first valid one would be wasted work.
__device__ __forceinline__ int spec_lanes(int nodes)
{
    return nodes <= kKeptNodes ? 16 : 64;
}
constexpr int kDraws = kMtN / 2; // 0-1 draws of a generator's block

// Runs request blockIdx.x's RRTConnect::solve loop for one slice.  Control
// flow is block-uniform: every thread holds the loop's variables and updates
// them identically; values one thread produces (the sample, the nearest
// node) reach the others through LDS.
template <int NT>
__global__ void __launch_bounds__(NT) plan_slice_kernel(SliceArgs A)
{
    __shared__ WaveTests s_tests[NT / 64];
    __shared__ double s_nodes[2][kDof * kKeptNodes];
    __shared__ uint32_t s_mt[kMtN];
    __shared__ double s_rstate[kDof];
    __shared__ double s_wd[NT / 64];
    __shared__ int s_wi[NT / 64];
    __shared__ double s_a[kDof], s_b[kDof], s_x[kDof]; // the step's motion and new state
    // the 0-1 draws of the generator's current 624-word block and, with `ahead`, of the next; s_mt is the last
    // block made, s_prev then the one before
    __shared__ double s_u[2 * kDraws];
    __shared__ uint32_t s_prev[kMtN];
    __shared__ int s_stop, s_n1, s_len;
    // speculative sampling steps: samples, motions, outcomes
    constexpr int kSpec = NT / 16 < 44 ? NT / 16 : 44; // their draws fit in one block
    static_assert(kSpec < 64 && kSpec * kDof <= NT && kSpec * kDof <= kDraws, "one lane an outcome, one thread a draw");
    __shared__ double s_samp[kSpec * kDof], s_ga[kSpec * kDof], s_gb[kSpec * kDof], s_gx[kSpec * kDof];
    __shared__ int s_open[kSpec], s_bad[kSpec], s_nm[kSpec], s_reach[kSpec], s_chk[kSpec], s_nd[kSpec], s_npos[kSpec];
    const int tid = threadIdx.x;
    const int64_t t0 = wall_clock64();
    const PlanCmd C = A.cmds[blockIdx.x];
    const GridView &g = C.grid;
    const RegionPtrs R = region_ptrs(C.region, C.cap);
    PlanState *st = R.state;
    // (selected, not indexed: an indexed local array lives in memory)
    auto tree = [&](int t) { return Tree{t ? R.tree_s[1] : R.tree_s[0], s_nodes[t], C.cap}; };
    auto parents = [&](int t) { return t ? R.parent[1] : R.parent[0]; };

    int mti, status, iteration, n0, n1, start_tree, tgi_start, grow_tree, phase, added, xmotion, path_len;
    int sampled_goals;
    int64_t steps, checks;
    if (C.init) {
        if (tid < 2 * kMaxEnds * kDof) R.ends[tid] = C.ends[tid];
        if (tid == 0) mt_seed_serial(s_mt, C.seed);
        if (tid < kDof) s_rstate[tid] = 0.0;
        mti = kMtN;
        status = OMPL_AMD_PLAN_RUNNING;
        iteration = 0;
        n0 = n1 = 0; // roots: the usable start states below, goal states in the loop
        sampled_goals = 0;
        start_tree = 1;
        tgi_start = 1;
        grow_tree = 0;
        phase = 0;
        added = xmotion = -1;
        path_len = 0;
        steps = checks = 0;
    } else {
        for (int i = tid; i < kMtN; i += NT) s_mt[i] = st->mt[i];
        if (tid < kDof) s_rstate[tid] = st->rstate[tid];
        mti = st->mti;
        status = st->status;
        iteration = st->iteration;
        n0 = st->n0;
        n1 = st->n1;
        start_tree = st->start_tree;
        tgi_start = st->tgi_start;
        grow_tree = st->grow_tree;
        phase = st->phase;
        added = st->added;
        xmotion = st->xmotion;
        path_len = st->path_len;
        sampled_goals = st->sampled_goals;
        steps = st->steps;
        checks = st->checks;
#pragma unroll
        for (int t = 0; t < 2; ++t)
            for (int i = tid; i < kDof * kKeptNodes; i += NT) {
                const int k = i / kKeptNodes, node = i % kKeptNodes;
                if (node < (t ? n1 : n0)) s_nodes[t][i] = R.tree_s[t][(int64_t)k * C.cap + node];
            }
    }
    __syncthreads();
    // words are consumed in pairs (mti is even); draw i is the i-th after the last one taken
    int pidx = mti / 2, cur = 0;
    bool ahead = false;
    auto make_draws = [&](int which) {
        for (int i = tid; i < kDraws; i += NT)
            s_u[which * kDraws + i] = canonical53(mt_temper(s_mt[2 * i]), mt_temper(s_mt[2 * i + 1]));
    };
    auto to_current = [&]() { // the block made ahead becomes the current one when that is used up
        if (ahead && pidx >= kDraws) {
            pidx -= kDraws;
            cur ^= 1;
            ahead = false;
        }
    };
    auto need_draws = [&](int need) { // need <= kDraws; whole block, a barrier before the draws are read
        to_current();
        if (!ahead && pidx + need > kDraws) {
            for (int i = tid; i < kMtN; i += NT) s_prev[i] = s_mt[i];
            mt_twist_block(s_mt); // reads the old words before its first barrier
            make_draws(cur ^ 1);
            ahead = true;
            to_current();
            __syncthreads();
        }
    };
    auto draw = [&](int i) {
        const int at = pidx + i;
        return s_u[at < kDraws ? cur * kDraws + at : (cur ^ 1) * kDraws + at - kDraws];
    };
    if (pidx < kDraws) make_draws(0);
    __syncthreads();
    if (C.init) {
        // PlannerInputStates::nextStart (Planner.cpp:228-256): the start
        // states in order; those in bounds and valid become the start tree's
        // roots
        for (int i = 0; i < C.n_starts; ++i) {
            if (endpoint_usable(g, R.ends + (size_t)i * kDof, s_x, s_tests) && n0 < C.cap) {
                if (tid < kDof) tree(0).set(tid, n0, s_x[tid]);
                if (tid == 0) R.parent[0][n0] = -1;
                ++n0;
            }
            __syncthreads(); // s_x is rewritten by the next state
        }
        if (n0 == 0) status = OMPL_AMD_PLAN_INVALID_START;
    }

    int done_here = 0;
    int64_t t_sample = 0, t_nearest = 0, t_check = 0, t_step = 0, c0 = 0, c1 = 0; // thread 0's timers
    while (status == OMPL_AMD_PLAN_RUNNING) {
        if (tid == 0) s_stop = done_here > 0 && wall_clock64() - t0 >= A.budget;
        __syncthreads();
        if (s_stop) break;
        // a step appends at most one node to one tree
        if (n0 >= C.cap || n1 >= C.cap) {
            status = OMPL_AMD_PLAN_TREE_FULL;
            break;
        }
        ++done_here;
        if (tid == 0) c0 = c1 = wall_clock64();
        // ---- speculative sampling steps.  A sampling step (phase 0) that is
        // TRAPPED changes neither tree, and the samples of the next steps are
        // the generator's next draws whatever happens, so the next m steps can
        // run at once, a few lanes each, against the current trees (step j
        // grows the start tree iff start_tree ^ (j & 1)); they are then taken in
        // order up to the first that is not TRAPPED, which is committed, and the
        // rest are dropped (their draws are not consumed).  Same steps, same
        // results as one at a time.  m stays within the iterations left.
        // (not while a goal state is due: the goal tree would change between
        // the steps)  The first connect step towards a node just added (phase 1)
        // is usually TRAPPED too, and then likewise changes nothing: it goes
        // before the sampling steps of a round as its step 0, which saves it a
        // pass of its own (64 requests over eight scenes 4.1 -> 3.3 ms).
        const bool goal_due = n1 == 0 || (sampled_goals < C.n_goals && sampled_goals < n1 / 2);
        const int lanes = spec_lanes(max(n0, n1));
        const int m = phase <= 1 && !goal_due ? min(min(kSpec, NT / lanes), C.max_iters - iteration) : 0;
        int gs = kTrapped;
        bool grown = false; // step 0 was a connect step that was not TRAPPED
        if (m >= 2) {
            const int first = phase; // steps before the sampling steps
            // whether step j's tgi.start (it grows the start tree)
            auto from_start = [&](int j, int start) { return j < first ? start : start ^ ((j - first) & 1); };
            const int start0 = start_tree; // in phase 1 tgi.start, too
            need_draws(kDof * (m - first));
            if (tid < kDof * m)
                s_samp[tid] = tid < kDof * first ? s_rstate[tid] : (kPi - -kPi) * draw(tid - kDof * first) + -kPi;
            __syncthreads();
            if (tid == 0) {
                c1 = wall_clock64();
                t_sample += c1 - c0;
            }
            const int wave = tid >> 6, lane = tid & 63;
            if (wave * 64 < m * lanes) {
                const int step = lanes == 64 ? wave : tid / 16, sub = tid & (lanes - 1), j = min(step, m - 1);
                const int st_j = from_start(j, start0);
                const int tree_j = st_j ? 0 : 1;
                const Tree Tj = tree(tree_j);
                double tgt[kDof];
#pragma unroll
                for (int k = 0; k < kDof; ++k) tgt[k] = s_samp[kDof * j + k];
                const int n_j = tree_j ? n1 : n0;
                Near best = scan_nearest(Tj, n_j, tgt, sub, lanes);
                best.share(lanes);
                if (tid == 0) {
                    const int64_t c2 = wall_clock64();
                    t_nearest += c2 - c1;
                }
                Steer S;
                S.run(Tj, n_j, best, tgt, C.maxd);
                double a[kDof], b[kDof];
#pragma unroll
                for (int k = 0; k < kDof; ++k) {
                    a[k] = st_j ? S.nst[k] : S.x[k];
                    b[k] = st_j ? S.x[k] : S.nst[k];
                }
                const int nd = valid_segment_count<kDof>(a, b, C.lvs, C.factor);
                // no progress, or too many segments: TRAPPED without a check
                const int npos = S.moved && nd <= kMaxSegments ? StepMotion::positions(nd, !st_j) : 0;
                if (sub == 0 && step < m) {
#pragma unroll
                    for (int k = 0; k < kDof; ++k) {
                        s_ga[kDof * j + k] = a[k];
                        s_gb[kDof * j + k] = b[k];
                        s_gx[kDof * j + k] = S.x[k];
                    }
                    s_nm[j] = S.nm;
                    s_reach[j] = S.reach ? 1 : 0;
                    s_chk[j] = S.moved ? 1 : 0;
                    s_nd[j] = nd;
                    s_npos[j] = npos;
                    s_bad[j] = 0;
                }
                // the steps' LDS writes before the wave's reads
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const StepMotion M{s_ga + kDof * j, s_gb + kDof * j, s_gx + kDof * j, nd, step < m ? npos : 0, !st_j};
                const uint64_t H = wave_ballot(wave_hit8(g, M, sub >> 3, s_tests[wave])) >> lane;
                if (sub == 0 && step < m) s_open[j] = npos > 0 && (lanes == 64 ? H : H & 0xffff) == 0;
            }
            __syncthreads();
            uint64_t open = wave_ballot(lane < m && s_open[min(lane, m - 1)] != 0);
            const uint64_t moved_steps = wave_ballot(lane < m && s_chk[min(lane, m - 1)] != 0);
            // the next positions of the open steps (those after the NT/64-th are
            // dropped with what follows them), the block's waves shared out
            int steps_here = m, checked = lanes / 8;
            if (open) {
                uint64_t more = open;
                int c = 0;
                for (; more && c < NT / 64; ++c) more &= more - 1;
                if (more) steps_here = lowest_bit(more);
                const int each = NT / 64 / c;
                if (wave < c * each) {
                    uint64_t rest = open;
                    for (int r = wave / each; r > 0; --r) rest &= rest - 1;
                    const int j = lowest_bit(rest);
                    const StepMotion M{s_ga + kDof * j, s_gb + kDof * j, s_gx + kDof * j, s_nd[j], s_npos[j],
                                       !from_start(j, start0)};
                    const int p = checked + 8 * (wave % each) + (lane >> 3);
                    if (wave_ballot(wave_hit8(g, M, p, s_tests[wave])) && lane == 0) s_bad[j] = 1;
                }
                checked += 8 * each;
                __syncthreads();
                if (steps_here < m) open &= ((uint64_t)1 << steps_here) - 1;
                open &= ~wave_ballot(lane < m && s_bad[min(lane, m - 1)] != 0);
            }
            // take the steps in order: those before the first open one together
            // (all TRAPPED), then that one
            phase = 0; // where a connect step that was TRAPPED leaves the loop
            for (int taken = 0; taken < steps_here;) {
                const int j = open ? lowest_bit(open) : steps_here;
                const uint64_t before = ((uint64_t)1 << j) - 1;
                const int samples = max(j, first) - max(taken, first);
                steps += j - taken;
                checks += __popcll(moved_steps & before & ~(((uint64_t)1 << taken) - 1));
                pidx += kDof * samples;
                start_tree ^= samples & 1; // RRTConnect.cpp:249
                iteration += j - taken;
                taken = j;
                if (j == steps_here) {
                    if (iteration >= C.max_iters) status = OMPL_AMD_PLAN_FAILED;
                    break;
                }
                const int st_j = start_tree;
                ++steps;
                ++checks; // an open step has moved
                const StepMotion M{s_ga + kDof * j, s_gb + kDof * j, s_gx + kDof * j, s_nd[j], s_npos[j], !st_j};
                const bool valid = block_check<NT>(g, M, checked, s_tests); // what is left of it
                if (j >= first) {
                    start_tree = !start_tree;
                    pidx += kDof; // this step's sample is consumed
                }
                ++taken;
                open &= open - 1;
                if (!valid) {
                    ++iteration;
                    if (iteration >= C.max_iters) {
                        status = OMPL_AMD_PLAN_FAILED;
                        break;
                    }
                    continue;
                }
                // commit step j: append its new state, then connect (phase 1)
                const int tree_j = st_j ? 0 : 1;
                const int last = append_step<NT>(tree(tree_j), parents(tree_j), tree_j ? n1 : n0, s_nm[j],
                                                 s_ga + kDof * j, s_gb + kDof * j, s_gx + kDof * j, s_nd[j], st_j != 0,
                                                 C.inter != 0);
                if (last < 0) {
                    status = OMPL_AMD_PLAN_TREE_FULL;
                    break;
                }
                xmotion = last;
                if (j < first) { // the solve loop goes on below
                    gs = s_reach[j] ? kReached : kAdvanced;
                    phase = 1;
                    grown = true;
                    break;
                }
                // rstate: the sample when reached, else the new state
                if (tid < kDof) s_rstate[tid] = s_reach[j] ? s_samp[kDof * j + tid] : s_gx[kDof * j + tid];
                added = last;
                tgi_start = start_tree;
                grow_tree = start_tree ? 0 : 1; // otherTree
                phase = 1;
                break;
            }
            if (tid == 0) t_check += wall_clock64() - c1;
            if (!grown) {
                if (tid == 0) t_step += wall_clock64() - c0;
                continue;
            }
        }
        if (!grown) {
            if (phase == 0) {
                // RRTConnect.cpp:247-250: pick the tree, flip startTree_
                grow_tree = start_tree ? 0 : 1;
                tgi_start = start_tree;
                start_tree = !start_tree;
                // RRTConnect.cpp:251-269: goal states (GoalStates, in order) --
                // every remaining one tried while the goal tree is empty
                // (nextGoal(ptc)), else one while fewer than half the goal tree's
                // size have been handed out (nextGoal())
                if (n1 == 0 || sampled_goals < n1 / 2) {
                    const bool empty = n1 == 0;
                    while (sampled_goals < C.n_goals) {
                        const int goal = sampled_goals++;
                        if (endpoint_usable(g, R.ends + (size_t)(kMaxEnds + goal) * kDof, s_x, s_tests)) {
                            if (n1 >= C.cap) {
                                status = OMPL_AMD_PLAN_TREE_FULL;
                            } else {
                                if (tid < kDof) tree(1).set(tid, n1, s_x[tid]);
                                if (tid == 0) R.parent[1][n1] = -1;
                                ++n1;
                            }
                            __syncthreads();
                            break;
                        }
                        __syncthreads();
                        if (!empty) break;
                    }
                    if (status == OMPL_AMD_PLAN_RUNNING && n1 == 0) status = OMPL_AMD_PLAN_INVALID_GOAL;
                    if (status != OMPL_AMD_PLAN_RUNNING) break;
                }
                // sampler_->sampleUniform(rstate): RNG::uniformReal(-pi, pi) per joint,
                // from the next seven draws
                need_draws(kDof);
                if (tid < kDof) s_rstate[tid] = (kPi - -kPi) * draw(tid) + -kPi;
                pidx += kDof;
                __syncthreads();
                if (tid == 0) {
                    c1 = wall_clock64();
                    t_sample += c1 - c0;
                }
            }

            // ---- growTree(tree, tgi, rmotion) (RRTConnect.cpp:116-196)
            double tgt[kDof];
#pragma unroll
            for (int k = 0; k < kDof; ++k) tgt[k] = s_rstate[k];
            const int nt = grow_tree ? n1 : n0;
            const Tree T = tree(grow_tree);
            const Near best = block_nearest<NT>(T, nt, tgt, s_wd, s_wi);
            if (tid == 0) {
                const int64_t c2 = wall_clock64();
                t_nearest += c2 - c1;
                c1 = c2;
            }
            Steer S;
            S.run(T, nt, best, tgt, C.maxd);
            if (S.moved) {
                // tgi.start ? checkMotion(nearest, dst) : isValid(dst) && checkMotion(dst, nearest)
                const bool from_start = tgi_start != 0;
                double a[kDof], b[kDof];
#pragma unroll
                for (int k = 0; k < kDof; ++k) {
                    a[k] = from_start ? S.nst[k] : S.x[k];
                    b[k] = from_start ? S.x[k] : S.nst[k];
                }
                const int nd = valid_segment_count<kDof>(a, b, C.lvs, C.factor);
                if (tid == 0) {
                    for (int k = 0; k < kDof; ++k) {
                        s_a[k] = a[k];
                        s_b[k] = b[k];
                        s_x[k] = S.x[k];
                    }
                }
                __syncthreads();
                ++checks;
                bool valid = false;
                if (nd <= kMaxSegments) { // longer motions are reported invalid
                    const StepMotion M{s_a, s_b, s_x, nd, StepMotion::positions(nd, !from_start), !from_start};
                    valid = !__syncthreads_or(wave_hit8(g, M, tid >> 3, s_tests[tid >> 6])) &&
                            block_check<NT>(g, M, NT / 8, s_tests);
                }
                if (valid) {
                    const int last = append_step<NT>(T, parents(grow_tree), grow_tree ? n1 : n0, S.nm, s_a, s_b, s_x,
                                                     nd, from_start, C.inter != 0);
                    if (last < 0) {
                        status = OMPL_AMD_PLAN_TREE_FULL;
                        break;
                    }
                    xmotion = last;
                    gs = S.reach ? kReached : kAdvanced;
                }
            }
            ++steps;
            if (tid == 0) t_check += wall_clock64() - c1;
        }

        // ---- solve loop (RRTConnect.cpp:245-330)
        bool end_iteration = false;
        if (phase == 0) {
            if (gs == kTrapped) {
                end_iteration = true;
            } else {
                added = xmotion;
                // if not reached, grow the other tree towards the added state
                if (gs != kReached && tid == 0)
                    for (int k = 0; k < kDof; ++k) s_rstate[k] = s_x[k];
                tgi_start = start_tree;
                grow_tree = start_tree ? 0 : 1; // otherTree
                phase = 1;
            }
        } else {
            if (phase == 1 && gs == kTrapped) tgi_start = !tgi_start;
            if (gs == kAdvanced) {
                phase = 2;
            } else if (gs == kReached) {
                // RRTConnect.cpp:301-330: step back once on the start side (or
                // the goal side at its root), then start chain reversed + goal chain
                int sm = tgi_start ? xmotion : added, gm = tgi_start ? added : xmotion;
                __syncthreads(); // a chain of intermediate states has parents from every wave
                if (tid == 0) {
                    const int32_t *ps = R.parent[0], *pg = R.parent[1];
                    if (ps[sm] >= 0) sm = ps[sm];
                    else gm = pg[gm];
                    int c = 0;
                    for (int m = sm; m >= 0; m = ps[m]) R.path_idx[c++] = m;
                    s_n1 = c;
                    for (int m = gm; m >= 0; m = pg[m]) R.path_idx[c++] = m;
                    s_len = c;
                }
                __syncthreads();
                const int c1 = s_n1, len = s_len;
                double *path = len <= A.path_rows ? C.path : R.path;
                for (int r = tid; r < len * kDof; r += NT) {
                    const int row = r / kDof, k = r - row * kDof;
                    path[r] = row < c1 ? R.tree_s[0][(int64_t)k * C.cap + R.path_idx[c1 - 1 - row]]
                                       : R.tree_s[1][(int64_t)k * C.cap + R.path_idx[row]];
                }
                path_len = len;
                status = OMPL_AMD_PLAN_SOLVED;
                ++iteration;
            } else {
                end_iteration = true;
            }
        }
        if (end_iteration) {
            phase = 0;
            ++iteration;
            if (iteration >= C.max_iters) status = OMPL_AMD_PLAN_FAILED;
        }
        if (tid == 0) t_step += wall_clock64() - c0;
    }

    __syncthreads();
    to_current();
    for (int i = tid; i < kMtN; i += NT) st->mt[i] = ahead ? s_prev[i] : s_mt[i];
    if (tid < kDof) st->rstate[tid] = s_rstate[tid];
    if (tid == 0) {
        st->mti = 2 * pidx;
        st->status = status;
        st->iteration = iteration;
        st->n0 = n0;
        st->n1 = n1;
        st->start_tree = start_tree;
        st->tgi_start = tgi_start;
        st->grow_tree = grow_tree;
        st->phase = phase;
        st->added = added;
        st->xmotion = xmotion;
        st->path_len = path_len;
        st->sampled_goals = sampled_goals;
        st->steps = steps;
        st->checks = checks;
        PlanOut &o = A.out[blockIdx.x];
        o.status = status;
        o.iteration = iteration;
        o.n0 = n0;
        o.n1 = n1;
        o.path_len = path_len;
        o.pad = 0;
        o.steps = steps;
        o.checks = checks;
        o.t_sample = t_sample;
        o.t_nearest = t_nearest;
        o.t_check = t_check;
        o.t_step = t_step;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
using Clock = std::chrono::steady_clock;

static double ms_since(Clock::time_point t0)
{
    return std::chrono::duration<double, std::milli>(Clock::now() - t0).count();
}

struct Planner {
    ompl_amd_plan_request req; // starts / goals point into `ends`
    // kMaxEnds start rows, then kMaxEnds goal rows (the region's layout)
    std::vector<double> ends = std::vector<double>((size_t)2 * kMaxEnds * kDof, 0.0);
    double maxd = 0.0;
    Clock::time_point t_submit, t_start, t_finish;
    // published: written and read under Server::mu only
    int status = OMPL_AMD_PLAN_QUEUED;
    int iterations = 0;
    int64_t nodes = 0;
    int64_t checks = 0;
    std::vector<double> path;
    bool started = false;
    bool cancel = false;
    bool env_held = false; // counted in the environment's server_users
    // server thread only
    size_t off = 0, bytes = 0; // region in the pool
    bool init = true;
    int64_t steps_seen = 0;
};

// Copies a request's start and goal states into the planner (the caller's
// lists need not outlive the submit): the lists, or start / goal when a list
// is empty.
static void take_endpoints(Planner &p)
{
    ompl_amd_plan_request &r = p.req;
    if (r.n_starts > 0) std::copy(r.starts, r.starts + (size_t)r.n_starts * kDof, p.ends.begin());
    else std::copy(r.start, r.start + kDof, p.ends.begin());
    if (r.n_goals > 0) std::copy(r.goals, r.goals + (size_t)r.n_goals * kDof, p.ends.begin() + (size_t)kMaxEnds * kDof);
    else std::copy(r.goal, r.goal + kDof, p.ends.begin() + (size_t)kMaxEnds * kDof);
    r.n_starts = r.n_starts > 0 ? r.n_starts : 1;
    r.n_goals = r.n_goals > 0 ? r.n_goals : 1;
    std::copy(p.ends.begin(), p.ends.begin() + kDof, r.start);
    std::copy(p.ends.begin() + (size_t)kMaxEnds * kDof, p.ends.begin() + (size_t)(kMaxEnds + 1) * kDof, r.goal);
    r.starts = p.ends.data();
    r.goals = p.ends.data() + (size_t)kMaxEnds * kDof;
}

// First-fit allocator over the device pool (offsets; neighbours coalesce).
struct PoolAlloc {
    std::map<size_t, size_t> free; // offset -> size
    void reset(size_t size)
    {
        free.clear();
        if (size) free[0] = size;
    }
    bool alloc(size_t bytes, size_t &off)
    {
        for (auto it = free.begin(); it != free.end(); ++it)
            if (it->second >= bytes) {
                off = it->first;
                const size_t rest = it->second - bytes;
                free.erase(it);
                if (rest) free[off + bytes] = rest;
                return true;
            }
        return false;
    }
    void release(size_t off, size_t bytes)
    {
        auto it = free.emplace(off, bytes).first;
        auto nx = std::next(it);
        if (nx != free.end() && it->first + it->second == nx->first) {
            it->second += nx->second;
            free.erase(nx);
        }
        if (it != free.begin()) {
            auto pv = std::prev(it);
            if (pv->first + pv->second == it->first) {
                pv->second += it->second;
                free.erase(it);
            }
        }
    }
};

struct Server {
    ompl_amd_server_config cfg;
    hipStream_t stream = nullptr;
    char *pool = nullptr;
    PoolAlloc alloc;
    // pinned, one per active request: the slice kernel reads and writes them in place
    PlanCmd *cmd_host = nullptr;
    PlanOut *out_host = nullptr;
    double *ends_host = nullptr; // [max_active][2 kMaxEnds][kDof]
    double *path_host = nullptr; // [max_active][path_rows][kDof]
    int path_rows = 0;
    int64_t budget_ticks = 0;

    std::mutex mu;
    std::condition_variable cv, done_cv;
    std::deque<int64_t> queue;
    std::unordered_map<int64_t, Planner *> reqs;
    std::vector<int64_t> active;
    int64_t next_id = 1;
    size_t used_bytes = 0;
    bool stop = false;
    std::thread th;
    std::atomic<int64_t> slices{0}, steps{0};
    int64_t phase_ticks[4] = {0, 0, 0, 0}; // sample, nearest, check, step (under mu)
    int64_t clock_khz = 0;
    std::string fault;
    // PRM requests: their own queue, worker thread and stream
    std::deque<int64_t> prm_queue;
    std::condition_variable prm_cv; // PRM arrivals and freed pool memory
    std::thread prm_th;
    hipStream_t prm_stream = nullptr;
    int prm_running = 0;

    void run();
    void run_prm();
    void admit_locked();
    void finish_locked(Planner *p, int status);
};

// Publishes a final status (caller holds mu), returns the region and
// releases the request's hold on its environment.
void Server::finish_locked(Planner *p, int status)
{
    p->status = status;
    p->t_finish = Clock::now();
    if (p->env_held) {
        p->req.env->server_users.fetch_sub(1);
        p->env_held = false;
    }
    if (p->bytes) {
        alloc.release(p->off, p->bytes);
        used_bytes -= p->bytes;
        p->bytes = 0;
        prm_cv.notify_all(); // a PRM request may be waiting for memory
    }
}

static size_t request_footprint(const ompl_amd_plan_request &r)
{
    return r.planner == OMPL_AMD_PLANNER_PRM ? prm_footprint(r.prm_samples, r.prm_k) : footprint(r.max_nodes);
}

// PRM requests, in arrival order, each once its roadmap's footprint is
// reserved in the pool (the roadmap itself is built in memory of its own).
void Server::run_prm()
{
    try {
        OA_HIP(hipSetDevice(device()));
        for (;;) {
            Planner *p = nullptr;
            {
                std::unique_lock<std::mutex> lk(mu);
                for (;;) {
                    if (stop) return;
                    if (!fault.empty()) return;
                    if (!prm_queue.empty()) {
                        Planner *q = reqs[prm_queue.front()];
                        const bool expired = q->req.deadline_ms > 0.0 && ms_since(q->t_submit) > q->req.deadline_ms;
                        if (q->cancel || expired) {
                            prm_queue.pop_front();
                            finish_locked(q, q->cancel ? OMPL_AMD_PLAN_CANCELLED : OMPL_AMD_PLAN_DEADLINE);
                            done_cv.notify_all();
                            continue;
                        }
                        const size_t fp = request_footprint(q->req);
                        size_t off = 0;
                        if (alloc.alloc(fp, off)) {
                            prm_queue.pop_front();
                            q->off = off;
                            q->bytes = fp;
                            used_bytes += fp;
                            q->status = OMPL_AMD_PLAN_RUNNING;
                            q->started = true;
                            q->t_start = Clock::now();
                            ++prm_running;
                            p = q;
                            break;
                        }
                    }
                    prm_cv.wait_for(lk, std::chrono::milliseconds(50));
                }
            }
            const ompl_amd_plan_request &r = p->req;
            const PrmQuery q = prm_query(r.env, r.start, r.goal, r.seed, 64, r.prm_samples, r.prm_k,
                                         r.longest_valid_segment, r.factor, prm_stream);
            std::lock_guard<std::mutex> lk(mu);
            p->iterations = 1;
            p->nodes = q.milestones;
            p->checks = q.candidate_edges;
            p->path = q.path;
            --prm_running;
            finish_locked(p, q.solved ? OMPL_AMD_PLAN_SOLVED : OMPL_AMD_PLAN_FAILED);
            done_cv.notify_all();
        }
    } catch (const std::exception &e) {
        std::lock_guard<std::mutex> lk(mu);
        if (fault.empty()) fault = e.what();
        for (auto &kv : reqs)
            if (kv.second->req.planner == OMPL_AMD_PLANNER_PRM && kv.second->status < OMPL_AMD_PLAN_SOLVED)
                finish_locked(kv.second, OMPL_AMD_PLAN_FAILED);
        prm_queue.clear();
        prm_running = 0;
        done_cv.notify_all();
    }
}

void Server::admit_locked()
{
    while (!queue.empty() && (int)active.size() < cfg.max_active) {
        const int64_t id = queue.front();
        Planner *p = reqs[id];
        const size_t fp = footprint(p->req.max_nodes);
        size_t off = 0;
        if (!alloc.alloc(fp, off)) break; // FIFO: the head waits for memory
        queue.pop_front();
        p->off = off;
        p->bytes = fp;
        used_bytes += fp;
        p->init = true;
        p->status = OMPL_AMD_PLAN_RUNNING;
        p->started = true;
        p->t_start = Clock::now();
        active.push_back(id);
    }
}

void Server::run()
{
    try {
        OA_HIP(hipSetDevice(device()));
        std::vector<Planner *> batch;
        std::vector<int64_t> batch_ids;
        std::vector<std::vector<double>> paths;
        for (;;) {
            batch.clear();
            batch_ids.clear();
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return stop || !queue.empty() || !active.empty(); });
                if (stop) return;
                bool notify = false;
                for (auto q = queue.begin(); q != queue.end();) {
                    Planner *p = reqs[*q];
                    if (p->req.deadline_ms > 0.0 && ms_since(p->t_submit) > p->req.deadline_ms) {
                        finish_locked(p, OMPL_AMD_PLAN_DEADLINE);
                        q = queue.erase(q);
                        notify = true;
                    } else {
                        ++q;
                    }
                }
                for (size_t i = 0; i < active.size();) {
                    Planner *p = reqs[active[i]];
                    const bool expired = p->req.deadline_ms > 0.0 && ms_since(p->t_submit) > p->req.deadline_ms;
                    if (p->cancel || expired) {
                        finish_locked(p, p->cancel ? OMPL_AMD_PLAN_CANCELLED : OMPL_AMD_PLAN_DEADLINE);
                        active.erase(active.begin() + (std::ptrdiff_t)i);
                        notify = true;
                    } else {
                        ++i;
                    }
                }
                admit_locked();
                for (int64_t id : active) {
                    batch.push_back(reqs[id]);
                    batch_ids.push_back(id);
                }
                if (notify) done_cv.notify_all();
            }
            if (batch.empty()) continue;
            const int n = (int)batch.size();
            for (int i = 0; i < n; ++i) {
                Planner &p = *batch[i];
                const Env &env = p.req.env->env;
                PlanCmd &c = cmd_host[i];
                c.grid = env.grid;
                c.region = pool + p.off;
                c.cap = p.req.max_nodes;
                c.max_iters = p.req.max_iters;
                c.maxd = p.maxd;
                c.lvs = p.req.longest_valid_segment;
                c.factor = p.req.factor;
                c.seed = p.req.seed;
                c.init = p.init ? 1 : 0;
                c.n_starts = p.req.n_starts;
                c.n_goals = p.req.n_goals;
                c.inter = p.req.intermediate_states ? 1 : 0;
                c.ends = ends_host + (size_t)i * 2 * kMaxEnds * kDof;
                c.path = path_host + (size_t)i * path_rows * kDof;
                if (p.init) std::copy(p.ends.begin(), p.ends.end(), ends_host + (size_t)i * 2 * kMaxEnds * kDof);
                p.init = false;
            }
            {
                ProfScope ps("serve_slice", stream);
                const SliceArgs args{cmd_host, out_host, path_rows, budget_ticks};
                if (cfg.block_threads == 1024)
                    hipLaunchKernelGGL(plan_slice_kernel<1024>, dim3(n), dim3(1024), 0, stream, args);
                else
                    hipLaunchKernelGGL(plan_slice_kernel<512>, dim3(n), dim3(512), 0, stream, args);
                OA_HIP(hipGetLastError());
            }
            OA_HIP(hipStreamSynchronize(stream));
            ++slices;
            // solution paths of the requests that solved in this slice
            paths.assign(n, {});
            bool copied = false;
            for (int i = 0; i < n; ++i) {
                const PlanOut &o = out_host[i];
                if (o.status != OMPL_AMD_PLAN_SOLVED || o.path_len <= 0) continue;
                paths[i].resize((size_t)o.path_len * kDof);
                if (o.path_len <= path_rows) {
                    const double *path = cmd_host[i].path;
                    std::copy(path, path + paths[i].size(), paths[i].begin());
                    continue;
                }
                const RegionPtrs Rp = region_ptrs(pool + batch[i]->off, batch[i]->req.max_nodes);
                OA_HIP(hipMemcpyAsync(paths[i].data(), Rp.path, paths[i].size() * sizeof(double),
                                      hipMemcpyDeviceToHost, stream));
                copied = true;
            }
            if (copied) OA_HIP(hipStreamSynchronize(stream));
            int64_t new_steps = 0;
            {
                std::lock_guard<std::mutex> lk(mu);
                bool notify = false;
                for (int i = 0; i < n; ++i) {
                    Planner *p = batch[i];
                    const PlanOut &o = out_host[i];
                    new_steps += o.steps - p->steps_seen;
                    phase_ticks[0] += o.t_sample;
                    phase_ticks[1] += o.t_nearest;
                    phase_ticks[2] += o.t_check;
                    phase_ticks[3] += o.t_step;
                    p->steps_seen = o.steps;
                    p->iterations = o.iteration;
                    p->nodes = (int64_t)o.n0 + o.n1;
                    p->checks = o.checks;
                    if (o.status == OMPL_AMD_PLAN_RUNNING) continue;
                    p->path.swap(paths[i]);
                    finish_locked(p, o.status);
                    active.erase(std::find(active.begin(), active.end(), batch_ids[i]));
                    notify = true;
                }
                if (notify) done_cv.notify_all();
            }
            steps += new_steps;
        }
    } catch (const std::exception &e) {
        std::lock_guard<std::mutex> lk(mu);
        fault = e.what();
        for (int64_t id : active) finish_locked(reqs[id], OMPL_AMD_PLAN_FAILED);
        for (int64_t id : queue) finish_locked(reqs[id], OMPL_AMD_PLAN_FAILED);
        for (int64_t id : prm_queue) finish_locked(reqs[id], OMPL_AMD_PLAN_FAILED);
        active.clear();
        queue.clear();
        prm_queue.clear();
        done_cv.notify_all();
        prm_cv.notify_all();
    }
}

static bool finished_status(int s)
{
    return s >= OMPL_AMD_PLAN_SOLVED;
}

// Caller holds Server::mu.
static void fill_result(const Planner &p, ompl_amd_plan_result *r)
{
    r->status = p.status;
    r->iterations = p.iterations;
    r->path_len = (int)(p.path.size() / kDof);
    r->tree_nodes = p.nodes;
    r->motion_checks = p.checks;
    auto ms = [](Clock::time_point a, Clock::time_point b) {
        return std::chrono::duration<double, std::milli>(b - a).count();
    };
    const bool done = finished_status(p.status);
    const Clock::time_point end = done ? p.t_finish : Clock::now();
    r->queued_ms = p.started ? ms(p.t_submit, p.t_start) : ms(p.t_submit, end);
    r->run_ms = p.started ? ms(p.t_start, end) : 0.0;
    r->latency_ms = ms(p.t_submit, end);
}

// ---------------------------------------------------------------------------
// plain path: host RRT-Connect, host nearest neighbours, one launch per check
// ---------------------------------------------------------------------------
struct HostTree {
    std::vector<double> s;
    std::vector<int> parent;
    int size() const { return (int)parent.size(); }
};

static int plain_grow(const Env &env, HostTree &t, bool start_tree, const double *target, double maxd, double lvs,
                      unsigned factor, bool inter, int &xmotion, double *xstate, int64_t &checks,
                      ThreadResources &tr)
{
    int nm = 0;
    double dmin = 0.0;
    for (int i = 0; i < t.size(); ++i) {
        double dist = 0.0;
        for (int k = 0; k < kDof; ++k) {
            const double diff = t.s[(size_t)i * kDof + k] - target[k];
            dist += diff * diff;
        }
        const double d = std::sqrt(dist);
        if (i == 0 || dmin > d) {
            nm = i;
            dmin = d;
        }
    }
    double ns[kDof]; // the tree may grow below
    std::copy(t.s.begin() + (size_t)nm * kDof, t.s.begin() + (size_t)(nm + 1) * kDof, ns);
    bool reach = true;
    double x[kDof];
    const double *dst = target;
    if (dmin > maxd) {
        bool equal = true;
        for (int k = 0; k < kDof; ++k) {
            x[k] = ns[k] + (target[k] - ns[k]) * (maxd / dmin);
            if (std::fabs(ns[k] - x[k]) > 2.220446049250313080847e-16 * 2.0) equal = false;
        }
        if (equal) return kTrapped;
        dst = x;
        reach = false;
    }
    auto check = [&](const double *a, const double *b) {
        Edge1 E;
        for (int k = 0; k < kDof; ++k) {
            E.a[k] = a[k];
            E.b[k] = b[k];
        }
        launch_motion_single(env.grid, E, lvs, factor, tr.pinned_dev, tr.stream);
        OA_HIP(hipStreamSynchronize(tr.stream));
        return tr.pinned[0] != 0;
    };
    bool valid;
    ++checks;
    if (start_tree) {
        valid = check(ns, dst);
    } else {
        State1 st;
        for (int k = 0; k < kDof; ++k) st.q[k] = dst[k];
        launch_validate_single(env.grid, st, tr.pinned_dev, tr.stream);
        OA_HIP(hipStreamSynchronize(tr.stream));
        valid = tr.pinned[0] != 0 && check(dst, ns);
    }
    if (!valid) return kTrapped;
    if (inter) {
        // getMotionStates(a, b, validSegmentCount(a, b), endpoints): states
        // 1 .. nd + 1 from the start tree, nd .. 0 from the goal tree
        const double *a = start_tree ? ns : dst, *b = start_tree ? dst : ns;
        const int seg = (int)valid_segment_count<kDof>(a, b, lvs, factor) + 1;
        int parent = nm;
        for (int r = 0; r < seg; ++r) {
            const int j = start_tree ? r + 1 : seg - 1 - r;
            for (int k = 0; k < kDof; ++k)
                t.s.push_back(j == 0 ? a[k] : (j == seg ? b[k] : a[k] + (b[k] - a[k]) * ((double)j / (double)seg)));
            t.parent.push_back(parent);
            parent = t.size() - 1;
        }
    } else {
        t.s.insert(t.s.end(), dst, dst + kDof);
        t.parent.push_back(nm);
    }
    xmotion = t.size() - 1;
    for (int k = 0; k < kDof; ++k) xstate[k] = dst[k];
    return reach ? kReached : kAdvanced;
}

// satisfiesBounds && isValid of one state (PlannerInputStates): one launch.
static bool plain_usable(const Env &env, const double *q, ThreadResources &tr)
{
    const double eps = 2.220446049250313080847e-16;
    for (int k = 0; k < kDof; ++k)
        if (q[k] - eps > kPi || q[k] + eps < -kPi) return false;
    State1 st;
    for (int k = 0; k < kDof; ++k) st.q[k] = q[k];
    launch_validate_single(env.grid, st, tr.pinned_dev, tr.stream);
    OA_HIP(hipStreamSynchronize(tr.stream));
    return tr.pinned[0] != 0;
}

// Plain PRM: the served PRM request's batch roadmap built on the host with one
// GPU launch and synchronisation per isValid / checkMotion call: samples from
// host std::mt19937 generators (the device sampler's streams), k-NN over the
// milestones in FP32 with the device search's distance and (distance, index)
// order, candidate edges checked from the lower milestone to the higher, host
// union-find, and the same shortest path.
static bool plain_prm(const ompl_amd_plan_request &req, const Env &env, ThreadResources &tr, std::vector<double> &out,
                      int64_t &milestones, int64_t &checks)
{
    const int streams = 64;
    const int samples = req.prm_samples > 0 ? req.prm_samples : 4096;
    const int k = req.prm_k > 0 ? req.prm_k : 10;
    const int64_t per = (samples + streams - 1) / streams;
    const int64_t n = 2 + per * streams;
    std::vector<double> smp((size_t)n * kDof);
    for (int d = 0; d < kDof; ++d) {
        smp[(size_t)d] = req.start[d];
        smp[(size_t)kDof + d] = req.goal[d];
    }
    for (int st = 0; st < streams; ++st) {
        std::mt19937 gen(req.seed + (uint32_t)st);
        std::uniform_real_distribution<> uni{0, 1};
        for (int64_t i = 0; i < per; ++i)
            for (int d = 0; d < kDof; ++d)
                smp[(size_t)(2 + st * per + i) * kDof + d] = (kPi - -kPi) * uni(gen) + -kPi;
    }
    std::vector<int32_t> ms;
    for (int64_t r = 0; r < n; ++r) {
        State1 q;
        for (int d = 0; d < kDof; ++d) q.q[d] = smp[(size_t)r * kDof + d];
        launch_validate_single(env.grid, q, tr.pinned_dev, tr.stream);
        OA_HIP(hipStreamSynchronize(tr.stream));
        if (tr.pinned[0] != 0) ms.push_back((int32_t)r);
    }
    const int64_t nv = (int64_t)ms.size();
    milestones = nv;
    checks = 0;
    if (nv < 2 || ms[0] != 0 || ms[1] != 1) return false;
    std::vector<double> nodes((size_t)nv * kDof);
    std::vector<float> f32((size_t)nv * kDof);
    for (int64_t i = 0; i < nv; ++i)
        for (int d = 0; d < kDof; ++d) {
            nodes[(size_t)i * kDof + d] = smp[(size_t)ms[(size_t)i] * kDof + d];
            f32[(size_t)i * kDof + d] = (float)nodes[(size_t)i * kDof + d];
        }
    // k + 1 nearest (the milestone itself among them), first k others kept
    const int64_t kk = std::min<int64_t>(k + 1, nv);
    std::vector<uint64_t> keys;
    std::vector<std::pair<float, int32_t>> cand((size_t)nv);
    for (int64_t i = 0; i < nv; ++i) {
        for (int64_t j = 0; j < nv; ++j) {
            float dist = 0.0f;
            for (int d = 0; d < kDof; ++d) {
                const float diff = f32[(size_t)j * kDof + d] - f32[(size_t)i * kDof + d];
                dist += diff * diff;
            }
            cand[(size_t)j] = {std::sqrt(dist), (int32_t)j};
        }
        std::partial_sort(cand.begin(), cand.begin() + kk, cand.end());
        int taken = 0;
        for (int64_t t = 0; t < kk && taken < k; ++t) {
            const int64_t j = cand[(size_t)t].second;
            if (j == i) continue;
            keys.push_back(((uint64_t)std::min(i, j) << 32) | (uint64_t)std::max(i, j));
            ++taken;
        }
    }
    std::sort(keys.begin(), keys.end());
    keys.erase(std::unique(keys.begin(), keys.end()), keys.end());
    checks = (int64_t)keys.size();
    std::vector<std::vector<int32_t>> nbr((size_t)nv);
    for (uint64_t key : keys) {
        const int32_t u = (int32_t)(key >> 32), v = (int32_t)(key & 0xffffffffu);
        Edge1 E;
        for (int d = 0; d < kDof; ++d) {
            E.a[d] = nodes[(size_t)u * kDof + d];
            E.b[d] = nodes[(size_t)v * kDof + d];
        }
        launch_motion_single(env.grid, E, req.longest_valid_segment, req.factor, tr.pinned_dev, tr.stream);
        OA_HIP(hipStreamSynchronize(tr.stream));
        if (tr.pinned[0] != 0) {
            nbr[(size_t)u].push_back(v);
            nbr[(size_t)v].push_back(u);
        }
    }
    std::vector<int64_t> off((size_t)nv + 1, 0);
    std::vector<int32_t> adj;
    for (int64_t i = 0; i < nv; ++i) {
        std::sort(nbr[(size_t)i].begin(), nbr[(size_t)i].end());
        adj.insert(adj.end(), nbr[(size_t)i].begin(), nbr[(size_t)i].end());
        off[(size_t)i + 1] = (int64_t)adj.size();
    }
    const std::vector<int32_t> path = roadmap_shortest_path(off, adj, nodes);
    for (int32_t v : path)
        out.insert(out.end(), nodes.begin() + (size_t)v * kDof, nodes.begin() + (size_t)(v + 1) * kDof);
    return !path.empty();
}

} // namespace ompl_amd

struct ompl_amd_server_s {
    ompl_amd::Server srv;
};

using namespace ompl_amd;

extern "C" {

int ompl_amd_server_create(const ompl_amd_server_config *cfg, ompl_amd_server *out)
{
    return guarded([&] {
        OA_REQUIRE(cfg && out, OMPL_AMD_ERR_ARG, "null argument");
        OA_REQUIRE(cfg->max_active >= 1 && cfg->max_active <= 65536, OMPL_AMD_ERR_ARG, "max_active in [1, 65536]");
        OA_REQUIRE(cfg->max_nodes >= 2, OMPL_AMD_ERR_ARG, "max_nodes >= 2");
        OA_REQUIRE(cfg->check_lanes_per_state == 0 || cfg->check_lanes_per_state == 7, OMPL_AMD_ERR_ARG,
                   "check_lanes_per_state must be 0 or 7 (the link layout)");
        const int co = cfg->check_obstacle_parts;
        OA_REQUIRE(co == 0 || co == 1 || co == 2 || co == 4 || co == 9, OMPL_AMD_ERR_ARG,
                   "check_obstacle_parts must be 0 (by motion length), 1, 2, 4 or 9");
        OA_REQUIRE(cfg->slice_us >= 0, OMPL_AMD_ERR_ARG, "slice_us must be >= 0");
        OA_REQUIRE(cfg->block_threads == 0 || cfg->block_threads == 512 || cfg->block_threads == 1024,
                   OMPL_AMD_ERR_ARG, "block_threads must be 0, 512 or 1024");
        ensure_init();
        auto *h = new ompl_amd_server_s();
        Server &S = h->srv;
        S.cfg = *cfg;
        S.cfg.check_lanes_per_state = 7;
        if (S.cfg.slice_us == 0) S.cfg.slice_us = 200;
        if (S.cfg.block_threads == 0) S.cfg.block_threads = 512; // 1,024 spills registers (measured slower)
        int rate_khz = 0;
        OA_HIP(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, device()));
        OA_REQUIRE(rate_khz > 0, OMPL_AMD_ERR_HIP, "device wall clock rate unavailable");
        S.clock_khz = rate_khz;
        S.budget_ticks = (int64_t)S.cfg.slice_us * rate_khz / 1000;
        if (S.budget_ticks < 1) S.budget_ticks = 1;
        OA_HIP(hipStreamCreateWithFlags(&S.stream, hipStreamNonBlocking));
        if (cfg->hbm_budget_bytes > 0) {
            hipError_t e = device_malloc(&S.pool, cfg->hbm_budget_bytes);
            if (e != hipSuccess) {
                (void)hipStreamDestroy(S.stream);
                delete h;
                fail(OMPL_AMD_ERR_NOMEM, "server pool of %zu bytes: %s", cfg->hbm_budget_bytes, hipGetErrorString(e));
            }
        }
        S.alloc.reset(cfg->hbm_budget_bytes);
        OA_HIP(hipHostMalloc((void **)&S.cmd_host, sizeof(PlanCmd) * cfg->max_active, hipHostMallocDefault));
        OA_HIP(hipHostMalloc((void **)&S.out_host, sizeof(PlanOut) * cfg->max_active, hipHostMallocDefault));
        OA_HIP(hipHostMalloc((void **)&S.ends_host, sizeof(double) * 2 * kMaxEnds * kDof * cfg->max_active,
                             hipHostMallocDefault));
        S.path_rows = std::max(1, std::min(kPathRows, (int)(kPathBytes / (sizeof(double) * kDof * cfg->max_active))));
        OA_HIP(hipHostMalloc((void **)&S.path_host, sizeof(double) * kDof * S.path_rows * cfg->max_active,
                             hipHostMallocDefault));
        OA_HIP(hipStreamCreateWithFlags(&S.prm_stream, hipStreamNonBlocking));
        S.th = std::thread([&S] { S.run(); });
        S.prm_th = std::thread([&S] { S.run_prm(); });
        *out = h;
    });
}

int ompl_amd_server_destroy(ompl_amd_server h)
{
    return guarded([&] {
        if (!h) return;
        Server &S = h->srv;
        {
            std::lock_guard<std::mutex> lk(S.mu);
            S.stop = true;
        }
        S.cv.notify_all();
        S.prm_cv.notify_all();
        if (S.th.joinable()) S.th.join();
        if (S.prm_th.joinable()) S.prm_th.join();
        for (auto &kv : S.reqs) {
            if (kv.second->env_held) kv.second->req.env->server_users.fetch_sub(1);
            delete kv.second;
        }
        // teardown: release everything even if one release reports an error
        (void)hipStreamSynchronize(S.stream);
        if (S.pool) (void)hipFree(S.pool);
        (void)hipHostFree(S.cmd_host);
        (void)hipHostFree(S.out_host);
        (void)hipHostFree(S.ends_host);
        (void)hipHostFree(S.path_host);
        (void)hipStreamDestroy(S.stream);
        (void)hipStreamSynchronize(S.prm_stream);
        (void)hipStreamDestroy(S.prm_stream);
        delete h;
    });
}

int ompl_amd_server_submit(ompl_amd_server h, const ompl_amd_plan_request *req, int64_t *id)
{
    return guarded([&] {
        OA_REQUIRE(h && req && id, OMPL_AMD_ERR_ARG, "null argument");
        OA_REQUIRE(req->env, OMPL_AMD_ERR_ARG, "request without environment");
        OA_REQUIRE(req->max_iters >= 1 && req->longest_valid_segment > 0.0 && req->factor >= 1, OMPL_AMD_ERR_ARG,
                   "bad request parameters");
        OA_REQUIRE(req->planner == OMPL_AMD_PLANNER_RRT_CONNECT || req->planner == OMPL_AMD_PLANNER_PRM,
                   OMPL_AMD_ERR_ARG, "unknown planner %d", req->planner);
        const Env &env = req->env->env;
        const bool prm = req->planner == OMPL_AMD_PLANNER_PRM;
        OA_REQUIRE(prm || env_stage_bytes(env.ns, env.nb) <= kPlanMaxEnvBytes, OMPL_AMD_ERR_ARG,
                   "environment too large for the server: %d spheres and %d boxes stage %zu bytes (limit %zu)",
                   env.ns, env.nb, env_stage_bytes(env.ns, env.nb), kPlanMaxEnvBytes);
        OA_REQUIRE(req->n_starts >= 0 && req->n_starts <= kMaxEnds && req->n_goals >= 0 && req->n_goals <= kMaxEnds,
                   OMPL_AMD_ERR_ARG, "a request lists at most %d start and %d goal states", kMaxEnds, kMaxEnds);
        OA_REQUIRE((req->n_starts == 0 || req->starts) && (req->n_goals == 0 || req->goals), OMPL_AMD_ERR_ARG,
                   "null start or goal list");
        OA_REQUIRE(!prm || (req->n_starts <= 1 && req->n_goals <= 1 && !req->intermediate_states), OMPL_AMD_ERR_ARG,
                   "PRM requests take one start and one goal state");
        Server &S = h->srv;
        auto *p = new Planner();
        p->req = *req;
        take_endpoints(*p);
        if (prm) {
            if (p->req.prm_samples <= 0) p->req.prm_samples = 4096;
            if (p->req.prm_k <= 0) p->req.prm_k = 10;
            OA_REQUIRE(p->req.prm_k <= 63 && p->req.prm_samples <= (1 << 24), OMPL_AMD_ERR_ARG,
                       "PRM request: prm_k <= 63 and prm_samples <= 2^24");
        }
        if (p->req.max_nodes <= 0 || p->req.max_nodes > S.cfg.max_nodes) p->req.max_nodes = S.cfg.max_nodes;
        if (p->req.max_nodes < 2) p->req.max_nodes = 2;
        if (p->req.max_nodes <= p->req.n_starts) {
            const int mn = p->req.max_nodes, ns = p->req.n_starts;
            delete p;
            fail(OMPL_AMD_ERR_ARG, "max_nodes %d cannot hold the %d start states and a step", mn, ns);
        }
        p->maxd = req->range > 0.0 ? req->range : 0.2 * 2.0 * kPi * std::sqrt(7.0);
        p->nodes = 2;
        p->t_submit = Clock::now();
        std::lock_guard<std::mutex> lk(S.mu);
        if (!S.fault.empty()) {
            delete p;
            fail(OMPL_AMD_ERR_HIP, "server stopped after a fault: %s", S.fault.c_str());
        }
        const int64_t rid = S.next_id++;
        S.reqs[rid] = p;
        if (request_footprint(p->req) > S.cfg.hbm_budget_bytes) {
            p->status = OMPL_AMD_PLAN_REJECTED;
            p->t_finish = p->t_submit;
        } else {
            p->req.env->server_users.fetch_add(1); // the environment must outlive the request
            p->env_held = true;
            if (prm) {
                S.prm_queue.push_back(rid);
                S.prm_cv.notify_all();
            } else {
                S.queue.push_back(rid);
            }
        }
        *id = rid;
        S.cv.notify_all();
    });
}

int ompl_amd_server_poll(ompl_amd_server h, int64_t id, ompl_amd_plan_result *res)
{
    return guarded([&] {
        OA_REQUIRE(h && res, OMPL_AMD_ERR_ARG, "null argument");
        Server &S = h->srv;
        std::lock_guard<std::mutex> lk(S.mu);
        auto it = S.reqs.find(id);
        OA_REQUIRE(it != S.reqs.end(), OMPL_AMD_ERR_ARG, "unknown request %lld", (long long)id);
        fill_result(*it->second, res);
    });
}

int ompl_amd_server_wait(ompl_amd_server h, int64_t id, double timeout_ms, ompl_amd_plan_result *res)
{
    return guarded([&] {
        OA_REQUIRE(h && res, OMPL_AMD_ERR_ARG, "null argument");
        Server &S = h->srv;
        std::unique_lock<std::mutex> lk(S.mu);
        auto it = S.reqs.find(id);
        OA_REQUIRE(it != S.reqs.end(), OMPL_AMD_ERR_ARG, "unknown request %lld", (long long)id);
        Planner *p = it->second;
        auto pred = [&] { return finished_status(p->status); };
        if (timeout_ms < 0) S.done_cv.wait(lk, pred);
        else S.done_cv.wait_for(lk, std::chrono::duration<double, std::milli>(timeout_ms), pred);
        fill_result(*p, res);
    });
}

int ompl_amd_server_path(ompl_amd_server h, int64_t id, double *out, int cap, int *n)
{
    return guarded([&] {
        OA_REQUIRE(h && n, OMPL_AMD_ERR_ARG, "null argument");
        Server &S = h->srv;
        std::lock_guard<std::mutex> lk(S.mu);
        auto it = S.reqs.find(id);
        OA_REQUIRE(it != S.reqs.end(), OMPL_AMD_ERR_ARG, "unknown request %lld", (long long)id);
        const auto &path = it->second->path;
        *n = (int)(path.size() / kDof);
        if (out && cap > 0)
            std::copy(path.begin(), path.begin() + std::min<size_t>(path.size(), (size_t)cap * kDof), out);
    });
}

int ompl_amd_server_cancel(ompl_amd_server h, int64_t id)
{
    return guarded([&] {
        OA_REQUIRE(h, OMPL_AMD_ERR_ARG, "null server");
        Server &S = h->srv;
        std::lock_guard<std::mutex> lk(S.mu);
        auto it = S.reqs.find(id);
        OA_REQUIRE(it != S.reqs.end(), OMPL_AMD_ERR_ARG, "unknown request %lld", (long long)id);
        Planner *p = it->second;
        p->cancel = true;
        if (p->status == OMPL_AMD_PLAN_QUEUED) {
            auto q = std::find(S.queue.begin(), S.queue.end(), id);
            if (q != S.queue.end()) S.queue.erase(q);
            auto qp = std::find(S.prm_queue.begin(), S.prm_queue.end(), id);
            if (qp != S.prm_queue.end()) S.prm_queue.erase(qp);
            S.finish_locked(p, OMPL_AMD_PLAN_CANCELLED);
            S.done_cv.notify_all();
        }
        S.cv.notify_all();
    });
}

int ompl_amd_server_release(ompl_amd_server h, int64_t id)
{
    return guarded([&] {
        OA_REQUIRE(h, OMPL_AMD_ERR_ARG, "null server");
        Server &S = h->srv;
        std::lock_guard<std::mutex> lk(S.mu);
        auto it = S.reqs.find(id);
        OA_REQUIRE(it != S.reqs.end(), OMPL_AMD_ERR_ARG, "unknown request %lld", (long long)id);
        OA_REQUIRE(finished_status(it->second->status), OMPL_AMD_ERR_ARG, "request %lld still running",
                   (long long)id);
        delete it->second;
        S.reqs.erase(it);
    });
}

int ompl_amd_server_stats(ompl_amd_server h, int64_t out[6])
{
    return guarded([&] {
        OA_REQUIRE(h && out, OMPL_AMD_ERR_ARG, "null argument");
        Server &S = h->srv;
        std::lock_guard<std::mutex> lk(S.mu);
        out[0] = S.slices.load();
        out[1] = S.steps.load();
        out[2] = (int64_t)S.active.size() + S.prm_running;
        out[3] = (int64_t)(S.queue.size() + S.prm_queue.size());
        out[4] = (int64_t)S.used_bytes;
        out[5] = (int64_t)S.cfg.hbm_budget_bytes;
    });
}

int ompl_amd_server_phase_us(ompl_amd_server h, double out[4])
{
    return guarded([&] {
        OA_REQUIRE(h && out, OMPL_AMD_ERR_ARG, "null argument");
        Server &S = h->srv;
        std::lock_guard<std::mutex> lk(S.mu);
        for (int i = 0; i < 4; ++i) out[i] = 1e3 * (double)S.phase_ticks[i] / (double)S.clock_khz;
    });
}

size_t ompl_amd_server_footprint(int max_nodes)
{
    return max_nodes >= 2 ? footprint(max_nodes) : 0;
}

int ompl_amd_plan_plain(const ompl_amd_plan_request *req, ompl_amd_plan_result *res, double *path, int cap,
                        int *path_len)
{
    return guarded([&] {
        OA_REQUIRE(req && res && req->env, OMPL_AMD_ERR_ARG, "null argument");
        const Clock::time_point t0 = Clock::now();
        const Env &env = req->env->env;
        ThreadResources &tr = thread_resources();
        if (req->planner == OMPL_AMD_PLANNER_PRM) {
            std::vector<double> out;
            int64_t nv = 0, checks = 0;
            const bool ok = plain_prm(*req, env, tr, out, nv, checks);
            const double ms = ms_since(t0);
            res->status = ok ? OMPL_AMD_PLAN_SOLVED : OMPL_AMD_PLAN_FAILED;
            res->iterations = 1;
            res->path_len = (int)(out.size() / kDof);
            res->tree_nodes = nv;
            res->motion_checks = checks;
            res->queued_ms = 0.0;
            res->run_ms = ms;
            res->latency_ms = ms;
            if (path_len) *path_len = res->path_len;
            if (path) std::copy(out.begin(), out.begin() + std::min<size_t>(out.size(), (size_t)cap * kDof), path);
            return;
        }
        OA_REQUIRE(req->planner == OMPL_AMD_PLANNER_RRT_CONNECT, OMPL_AMD_ERR_ARG, "unknown planner %d",
                   req->planner);
        std::mt19937 gen(req->seed);
        std::uniform_real_distribution<> uni{0, 1};
        const double maxd = req->range > 0.0 ? req->range : 0.2 * 2.0 * kPi * std::sqrt(7.0);
        OA_REQUIRE(req->n_starts >= 0 && req->n_starts <= kMaxEnds && req->n_goals >= 0 && req->n_goals <= kMaxEnds &&
                       (req->n_starts == 0 || req->starts) && (req->n_goals == 0 || req->goals),
                   OMPL_AMD_ERR_ARG, "bad start or goal list");
        const double *starts = req->n_starts > 0 ? req->starts : req->start;
        const double *goals = req->n_goals > 0 ? req->goals : req->goal;
        const int n_starts = req->n_starts > 0 ? req->n_starts : 1, n_goals = req->n_goals > 0 ? req->n_goals : 1;
        const bool inter = req->intermediate_states != 0;
        HostTree ts, tg;
        for (int i = 0; i < n_starts; ++i) // nextStart: usable start states become roots
            if (plain_usable(env, starts + (size_t)i * kDof, tr)) {
                ts.s.insert(ts.s.end(), starts + (size_t)i * kDof, starts + (size_t)(i + 1) * kDof);
                ts.parent.push_back(-1);
            }
        bool start_tree = true, solved = false;
        int it = 0, sampled_goals = 0;
        int status = ts.size() == 0 ? OMPL_AMD_PLAN_INVALID_START : OMPL_AMD_PLAN_RUNNING;
        int64_t checks = 0;
        double rstate[kDof], xstate[kDof];
        std::vector<double> out;
        for (it = 0; it < req->max_iters && !solved && status == OMPL_AMD_PLAN_RUNNING; ++it) {
            if (req->deadline_ms > 0.0 && ms_since(t0) > req->deadline_ms) break;
            HostTree &tree = start_tree ? ts : tg;
            bool tgi_start = start_tree;
            start_tree = !start_tree;
            HostTree &other = start_tree ? ts : tg;
            if (tg.size() == 0 || sampled_goals < tg.size() / 2) { // goal states, as the served planner
                const bool empty = tg.size() == 0;
                while (sampled_goals < n_goals) {
                    const double *q = goals + (size_t)(sampled_goals++) * kDof;
                    if (plain_usable(env, q, tr)) {
                        tg.s.insert(tg.s.end(), q, q + kDof);
                        tg.parent.push_back(-1);
                        break;
                    }
                    if (!empty) break;
                }
                if (tg.size() == 0) {
                    status = OMPL_AMD_PLAN_INVALID_GOAL;
                    break;
                }
            }
            for (int k = 0; k < kDof; ++k) rstate[k] = (kPi - -kPi) * uni(gen) + -kPi;
            int xm = -1;
            int gs = plain_grow(env, tree, tgi_start, rstate, maxd, req->longest_valid_segment, req->factor, inter, xm,
                                xstate, checks, tr);
            if (gs == kTrapped) continue;
            const int added = xm;
            if (gs != kReached)
                for (int k = 0; k < kDof; ++k) rstate[k] = xstate[k];
            tgi_start = start_tree;
            int gsc = plain_grow(env, other, tgi_start, rstate, maxd, req->longest_valid_segment, req->factor, inter,
                                 xm, xstate, checks, tr);
            if (gsc == kTrapped) tgi_start = !tgi_start;
            while (gsc == kAdvanced)
                gsc = plain_grow(env, other, tgi_start, rstate, maxd, req->longest_valid_segment, req->factor, inter,
                                 xm, xstate, checks, tr);
            if (gsc != kReached) continue;
            int sm = tgi_start ? xm : added, gm = tgi_start ? added : xm;
            if (ts.parent[sm] >= 0) sm = ts.parent[sm];
            else gm = tg.parent[gm];
            std::vector<int> c1, c2;
            for (int m = sm; m >= 0; m = ts.parent[m]) c1.push_back(m);
            for (int m = gm; m >= 0; m = tg.parent[m]) c2.push_back(m);
            for (int i = (int)c1.size() - 1; i >= 0; --i)
                out.insert(out.end(), ts.s.begin() + (size_t)c1[i] * kDof, ts.s.begin() + (size_t)(c1[i] + 1) * kDof);
            for (int m : c2) out.insert(out.end(), tg.s.begin() + (size_t)m * kDof, tg.s.begin() + (size_t)(m + 1) * kDof);
            solved = true;
        }
        const double ms = ms_since(t0);
        res->status = solved ? OMPL_AMD_PLAN_SOLVED
                      : status != OMPL_AMD_PLAN_RUNNING
                          ? status
                          : ((req->deadline_ms > 0.0 && ms > req->deadline_ms) ? OMPL_AMD_PLAN_DEADLINE
                                                                                  : OMPL_AMD_PLAN_FAILED);
        res->iterations = it;
        res->path_len = (int)(out.size() / kDof);
        res->tree_nodes = ts.size() + tg.size();
        res->motion_checks = checks;
        res->queued_ms = 0.0;
        res->run_ms = ms;
        res->latency_ms = ms;
        if (path_len) *path_len = res->path_len;
        if (path) std::copy(out.begin(), out.begin() + std::min<size_t>(out.size(), (size_t)cap * kDof), path);
    });
}

} // extern "C"
