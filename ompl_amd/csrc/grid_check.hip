// State validity, motion validation, lastValid and state lists over an
// environment's cell grid (grid.hpp).
//
// A state is 28 sphere centres; the base link's four never move and are
// decided when the environment is made.  Each of the other six links looks up
// the cell of its second sphere: its clearance may spare the whole link or all
// but its last sphere; else the cells of the other three are looked up as well.
// Only spheres in a cell that some obstacle's surface passes near are tested,
// against the obstacles the cell lists, with the exact predicate
// (arm_device.hpp), so results are the same bits as a test against every
// obstacle.  On the 128 + 128 obstacle scene that is 6 to 24 reads of a 1 MiB
// table and a few exact tests per state where the full test has 28 x 256.
//
// A walk need not look at every position either: the clearances of a state and
// the joints' levers say how many positions before and after it are certainly
// valid (with margins of 1e-4 m and more for the rounding of states and
// centres), so of a roadmap's edges, 126 positions long, 31 are looked at and
// then 32 more on average (wave_edges).
//
// Lane mapping: one state per lane (no redundant forward kinematics: the
// fastest where there are states enough), or eight lanes per state, one link
// each (a third of the latency, twice the instructions).
//
// Measured against the kernels that tested every obstacle, in the launch shapes
// the library starts with: 65,536 states, 64 spheres 35.7 -> 8.7 us; 16,384
// edges, 16 + 16 obstacles, checked counts 385 -> 44 us; 4,099 edges' lastValid
// 110 -> 24 us; 61 edges, 128 + 128 obstacles 38 -> 8.8 us.  Against shapes
// tuned for the scene: 16,384 edges, 128 + 128 obstacles 31 -> 19.0 us on one
// stream, 12.6 -> 8.3 us a batch on four; 16 + 16 obstacles 77 -> 39 us (no
// counts).  Large batches are bound by VALU instructions (about 1,100 a wave of
// 64 states, half of them the forward kinematics): 836,000 roadmap edges, 64
// spheres 4.8 ms with every position looked at, 1.3 ms with the gaps.  Small
// ones are bound by the chain of dependent reads (counts, record, cells, cells,
// obstacles), by fetching the code once and by the launches: a kernel that only
// walked what the one before had left cost 3 to 4 us, so the survivors' kernel
// walks its own leftovers (16,384 dense edges 22.2 -> 19.0 us, 11.3 -> 8.3 on
// four streams) and a one-launch batch finds its own long items (61 edges 11.7
// -> 8.8 us).
#include <hip/hip_runtime.h>

#include <climits>

#include "check_device.hpp"
#include "checker.hpp"
#include "grid_device.hpp"
#include "motion_device.hpp"
#include "walk_device.hpp"

namespace ompl_amd {

// ---------------------------------------------------------------------------
// validity
// ---------------------------------------------------------------------------
template <int LANES, typename T>
__global__ void __launch_bounds__(256) grid_validate_kernel(GridView g, const T *__restrict__ q_soa, int64_t n,
                                                            uint8_t *__restrict__ out)
{
    __shared__ WaveTests tests[4];
    const int64_t st = (xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x) / LANES;
    const bool live = st < n;
    bool hit;
    if constexpr (LANES == 1) {
        float q[kDof];
        load_config(q_soa, n, st, live, q);
        hit = state_hit1(g, q, live, tests[threadIdx.x >> 6]);
    } else {
        const int j = min((int)threadIdx.x & 7, kDof - 1);
        hit = state_hit8(g, (float)q_soa[(int64_t)j * n + (live ? st : 0)], live, tests[threadIdx.x >> 6]);
    }
    const uint64_t H = fold_groups<LANES>(wave_ballot(hit));
    const int lane = lane_id();
    if (live && lane % LANES == 0) out[st] = ((H >> lane) & 1) ? 0 : 1;
}

// ---------------------------------------------------------------------------
// motions, lastValid, state lists
// ---------------------------------------------------------------------------
// What is walked: kBisect, an edge's positions 1 .. nd-1 in bisection order
// (position 0, its s2, first where the walk starts there); kSequence, positions
// 1 .. nd in order, nd being s2 (DiscreteMotionValidator.cpp:48-91); kList, the
// states of a precomputed list in order (SpaceInformation.cpp:288-299).
enum class Walk { kBisect, kSequence, kList };

// Items with more than kLongWalk positions are long: walked by many blocks
// together, each every so-manyth 256 of its positions.  A long item has a word
// for the lowest position found invalid (INT_MAX minus it, 0: none) and a
// ticket; the last block to finish it writes its result.
constexpr int kLongWalk = 16384;
// Blocks that look for long items beside up to kWideItems blocks of an item each.
constexpr int kHelpers = 256;

struct GridWalkArgs {
    GridView g;
    MotionArgs m;
    double *last_t;    // kSequence
    const double *q;   // kList: dof-major states
    int64_t n_states;
    const int64_t *offsets;
    int32_t *rest;      // [cap] lists of a wave each: whether the item is unfinished (listing
                        // them would take a device-wide atomic each: on one address they
                        // are 6 ns apart, 60 us for 10,000)
    int32_t *long_slot; // [cap] long items
    int32_t *long_bad;  // [cap]
    int32_t *ticket;    // [cap]
    int32_t *wide_bad;  // [kWideItems] by item, zero between batches
    int32_t *wide_ticket;
    int32_t *counts;    // [0] survivors, [1] long items; zero at the batch's start
    int32_t *next;      // the set the next batch uses, cleared by the first kernel after the s2 pass
};

// One item: its id (edge or list) and what is needed to make its states.
template <Walk MODE>
struct Item {
    int64_t id;
    double a[kDof], b[kDof];
    int64_t lo;
    int nd, total; // positions are below `total`
    __device__ __forceinline__ void edge(const MotionArgs &A, int64_t e)
    {
        id = e;
#pragma unroll
        for (int j = 0; j < kDof; ++j) {
            a[j] = A.a[(int64_t)j * A.n + e];
            b[j] = A.b[(int64_t)j * A.n + e];
        }
        nd = valid_segment_count<kDof>(a, b, A.lvs, A.factor);
        total = MODE == Walk::kBisect ? max(nd, 1) : max(nd, 1) + 1;
    }
    // As edge() for a wave-uniform e.  The edges, as a survivor's record below,
    // were written by earlier kernels, so they are read into scalar registers (28
    // vector registers fewer: a wave more per SIMD).
    __device__ __forceinline__ void one_edge(const MotionArgs &A, int e_any)
    {
        using Const = const __attribute__((address_space(4))) double;
        const int e = __builtin_amdgcn_readfirstlane(e_any);
        id = e;
#pragma unroll
        for (int j = 0; j < kDof; ++j) {
            a[j] = ((Const *)A.a)[(int64_t)j * A.n + e];
            b[j] = ((Const *)A.b)[(int64_t)j * A.n + e];
        }
        nd = valid_segment_count<kDof>(a, b, A.lvs, A.factor);
        total = MODE == Walk::kBisect ? max(nd, 1) : max(nd, 1) + 1;
    }
    // slot is wave-uniform
    __device__ __forceinline__ void survivor(const MotionArgs &A, int slot_any)
    {
        using Const = const __attribute__((address_space(4))) double;
        const int slot = __builtin_amdgcn_readfirstlane(slot_any);
        Const *ab = (Const *)(A.surv_ab + (int64_t)slot * 2 * kDof);
#pragma unroll
        for (int j = 0; j < kDof; ++j) {
            a[j] = ab[j];
            b[j] = ab[kDof + j];
        }
        nd = A.surv_nd[slot];
        id = A.list[slot];
        total = MODE == Walk::kBisect ? max(nd, 1) : max(nd, 1) + 1;
    }
    __device__ __forceinline__ bool nd_too_many() const { return MODE != Walk::kList && nd > kMaxSegments; }
    __device__ __forceinline__ void list(const GridWalkArgs &A, int64_t l)
    {
        id = l;
        lo = min(max(A.offsets[l], (int64_t)0), A.n_states);
        total = (int)(max(min(A.offsets[l + 1], A.n_states), lo) - lo);
    }
    __device__ __forceinline__ void state(const GridWalkArgs &A, int p, float q[kDof]) const
    {
        if (MODE == Walk::kBisect) {
            walk_state(a, b, nd, p, q);
        } else if (MODE == Walk::kSequence) {
            if (p >= total - 1) {
#pragma unroll
                for (int j = 0; j < kDof; ++j) q[j] = (float)b[j];
            } else {
                interpolate_f32<kDof>(a, b, (double)p / (double)nd, q);
            }
        } else {
#pragma unroll
            for (int j = 0; j < kDof; ++j) q[j] = (float)A.q[(int64_t)j * A.n_states + lo + p];
        }
    }
    // Result from the lowest invalid position (INT_MAX: none); one lane.
    __device__ __forceinline__ void result(const GridWalkArgs &A, int bad) const
    {
        const bool ok = bad == INT_MAX;
        A.m.out[id] = ok ? 1 : 0;
        if (MODE == Walk::kBisect) {
            if (A.m.checked) A.m.checked[id] = ok ? total : bad + 1;
        } else if (MODE == Walk::kSequence) {
            // an interior position j: (j - 1) / nd; s2: (nd - 1) / nd
            if (!ok) A.last_t[id] = bad < total - 1 ? (double)(bad - 1) / (double)nd : (double)(nd - 1) / (double)nd;
        } else {
            if (A.m.checked) A.m.checked[id] = ok ? -1 : bad;
        }
    }
};

// Lowest invalid of the positions base + lane below `total` (one state per
// lane), or INT_MAX; wave-uniform.
template <Walk MODE>
__device__ __forceinline__ int wave_walk(const GridWalkArgs &A, const Item<MODE> &I, int base, int total,
                                         WaveTests *tests)
{
    if (base >= total) return INT_MAX;
    const int p = base + lane_id();
    const bool live = p < total;
    float q[kDof];
    I.state(A, live ? p : base, q);
    const uint64_t H = wave_ballot(state_hit1(A.g, q, live, tests[threadIdx.x >> 6]));
    return H ? base + lowest_bit(H) : INT_MAX; // wave-uniform
}

__device__ __forceinline__ int known_bad(const int32_t *p)
{
    return INT_MAX - __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What the waves of a block tell each other after a round, twice over so that
// one barrier a round is enough.
struct Rounds {
    int bad[2][4];
    int known[2];
};

// The walk of one item by a block: its positions below `end` from `first` on, a
// block's at a time, `step` apart.  The kernels below have one call of it each:
// the code of a state check is 10 KB, and a short launch waits for every line of it.
// known: a long item's word (else null), which ends the walk once an earlier
// position is known invalid.  Returns the lowest invalid position seen or
// INT_MAX, uniform over the walkers.
template <Walk MODE>
__device__ __forceinline__ int walk_item(const GridWalkArgs &A, const Item<MODE> &I, int64_t first, int end,
                                         int64_t step, const int32_t *known, Rounds &R, int &turn, WaveTests *tests)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int64_t round = first;;) {
        const int64_t base = round + wave * 64;
        const int b = wave_walk<MODE>(A, I, (int)min(base, (int64_t)INT_MAX), end, tests);
        if (lane_id() == 0) R.bad[turn][wave] = b;
        if (threadIdx.x == 0) R.known[turn] = known ? known_bad(known) : INT_MAX;
        __syncthreads();
        const int found = __builtin_amdgcn_readfirstlane(
            min(min(R.bad[turn][0], R.bad[turn][1]), min(R.bad[turn][2], R.bad[turn][3])));
        const int earlier = __builtin_amdgcn_readfirstlane(R.known[turn]);
        turn ^= 1;
        round += step;
        if (found != INT_MAX || round >= end || earlier < round) return found; // block-uniform
    }
}

// A block's share of a long item is done (one thread); `blocks` of them.
template <Walk MODE>
__device__ __forceinline__ void finish_long(const GridWalkArgs &A, const Item<MODE> &I, int b, int32_t *bad,
                                            int32_t *ticket, int blocks)
{
    if (b != INT_MAX) atomicMax(bad, INT_MAX - b);
    __threadfence(); // the minimum is made before the ticket is taken
    if (atomicAdd(ticket, 1) != blocks - 1) return;
    __threadfence();
    I.result(A, known_bad(bad));
    *bad = 0; // as the next batch finds them
    *ticket = 0;
}

// Lists a long item (one lane).
__device__ __forceinline__ void list_long(const GridWalkArgs &A, int slot)
{
    const int l = atomicAdd(&A.counts[1], 1);
    A.long_slot[l] = slot;
    A.long_bad[l] = 0;
    A.ticket[l] = 0;
}

__device__ __forceinline__ void clear_next(const GridWalkArgs &A)
{
    if (blockIdx.x == 0 && threadIdx.x < 2) A.next[threadIdx.x] = 0;
}

// s2 of every edge; survivors (s2 valid, 2 <= nd) go to the list.  One lane
// per edge: large batches.
__global__ void __launch_bounds__(256) grid_endpoint1_kernel(GridWalkArgs A)
{
    __shared__ WaveTests tests[4];
    const MotionArgs &M = A.m;
    const int64_t e = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const bool live = e < M.n;
    float q[kDof];
    load_config(M.b, M.n, e, live, q);
    const uint64_t H = wave_ballot(state_hit1(A.g, q, live, tests[threadIdx.x >> 6]));
    int m = 0;
    double a[kDof], b[kDof];
    const bool survivor = endpoint_finish<1>(M, e, live, H, m, a, b);
    const int slot = append_survivor(M, e, survivor, m, a, b);
    if (survivor && m > kLongWalk) list_long(A, slot);
}

// As above with eight lanes per edge: lane j reads joint j of both ends (two
// reads in flight in place of 7 and then 14) and writes it to a survivor's
// record.
__global__ void __launch_bounds__(256) grid_endpoint8_kernel(GridWalkArgs A)
{
    __shared__ WaveTests tests[4];
    __shared__ int blk_count, blk_base;
    const MotionArgs &M = A.m;
    if (threadIdx.x == 0) blk_count = 0;
    const int64_t e = (xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x) >> 3;
    const bool live = e < M.n;
    const int lane = lane_id(), j = lane & 7;
    const int64_t at = (int64_t)min(j, kDof - 1) * M.n + (live ? e : 0);
    const double bj = M.b[at], aj = M.a[at];
    const bool hit = state_hit8(A.g, (float)bj, live, tests[threadIdx.x >> 6]);
    const uint64_t H = fold_groups<8>(wave_ballot(hit));
    const bool bad = ((H >> (lane & 56)) & 1) != 0;
    int nd = 0;
    if (wave_ballot(live && !bad)) {
        const double diff = aj - bj, sq = diff * diff;
        double dist2 = 0.0;
#pragma unroll
        for (int i = 0; i < kDof; ++i) dist2 += __shfl(sq, (lane & 56) + i);
        nd = segments_of(dist2, M.lvs, M.factor);
    }
    const bool survivor = live && !bad && nd >= 2 && nd <= kMaxSegments;
    if (live && j == 0) {
        M.out[e] = !bad && nd <= kMaxSegments ? 1 : 0; // a survivor's until the walk finds an invalid position
        if (M.checked && !survivor) M.checked[e] = !bad && nd > kMaxSegments ? 0 : 1;
    }
    // the block's survivors take consecutive slots
    const uint64_t sm = wave_ballot(survivor && j == 0);
    __syncthreads();
    int woff = 0;
    if (sm) {
        if (lane == lowest_bit(sm)) woff = atomicAdd(&blk_count, __popcll(sm));
        woff = __shfl(woff, lowest_bit(sm));
    }
    __syncthreads();
    if (blk_count == 0) return; // block-uniform
    if (threadIdx.x == 0) blk_base = atomicAdd(M.list_count, blk_count);
    __syncthreads();
    if (survivor) {
        const int slot = blk_base + woff + __popcll(sm & (((uint64_t)1 << (lane & 56)) - 1));
        if (j == 0) {
            M.list[slot] = (int32_t)e;
            M.surv_nd[slot] = nd;
            if (nd - 1 > kLongWalk) list_long(A, slot);
        }
        if (j < kDof) {
            double *ab = M.surv_ab + (int64_t)slot * 2 * kDof;
            ab[j] = aj;
            ab[kDof + j] = bj;
        }
    }
}

// A wave's view of the edges it walks (LDS): a ring of edges, and a ring of the
// states to look at, each an edge's slot and an index along it.
struct WaveEdges {
    static constexpr int kEdges = 8, kStates = 256;
    struct Edge {
        double ab[2 * kDof];
        int32_t id, nd;
        int bad; // lowest position found invalid
        int end; // the edge is done when so many states have been looked at
    } edge[kEdges];
    int state[kStates]; // slot << 24 | index
};
struct BlockEdges {
    WaveEdges wave[4];
    int looked[4], held[4]; // of the waves' rings, while the block shares them
};

// The first 2^levels - 1 positions of the bisection are a complete binary tree
// over the edge's interior: in order, the s-th of them (from 1) is the one with
// this number (root 1).
__device__ __forceinline__ int heap_of_slot(int s, int levels)
{
    const int up = __builtin_ctz(s);
    return (1 << (levels - 1 - up)) + (s >> (up + 1));
}

// How fast the spheres of links 1 .. 6 move along an edge: a joint moves a
// sphere by at most its angle times the sphere's distance from its axis, 0.3 m a
// link between them and 0.2625 m on the last; an even joint turns its own link
// about itself.  An edge with a coordinate beyond 16 rad, where rounding to FP32
// would eat into the margin, gets no clearance.
// `need` positions are worth looking closer for.
__device__ __forceinline__ void edge_speeds(const double a[kDof], const double b[kDof], int nd, float need,
                                            Speeds &sp)
{
    float d[kDof];
    bool plain = true;
#pragma unroll
    for (int j = 0; j < kDof; ++j) {
        d[j] = (float)fabs(b[j] - a[j]);
        plain = plain && fabs(a[j]) <= 16.0 && fabs(b[j]) <= 16.0;
    }
    float most = 0.0f;
#pragma unroll
    for (int i = 1; i < kDof; ++i) {
        float v = 0.0f;
#pragma unroll
        for (int j = 0; j <= i; ++j) {
            const int links = (j & 1) ? i - j : i - j - 1;
            if (links >= 0) v += d[j] * (0.3f * (float)links + 0.2625f);
        }
        v = v * 1.0001f + 1e-6f; // metres from end to end
        most = fmaxf(most, v);
        sp.steps[i - 1] = plain ? (float)nd / (v * kClearUnits) : 0.0f;
    }
    const uint32_t units = plain ? (uint32_t)(most * kClearUnits * (need / (float)max(nd, 1))) : 0u;
    sp.far = kFarUnits + units;
    sp.near = kClearReachUnits + units;
}

// A wave's share of the survivors (kBisect) or edges (kSequence): pairs first,
// first + step, ...  It looks at 31 evenly spread positions of two edges at once
// (the first 31 of the bisection; beside them s1, for its clearance, or s2): how
// far the arm can move from each before a sphere could touch anything says which
// of the positions between them are certainly valid.  Only the others are looked at, 64 at a
// time, from as many edges as that takes.  A wave that has taken its last pair
// waits for the block's others, and they look at what is left together: a pair
// of long edges leaves ten passes, which would be the launch's end (16,384
// edges, 16 + 16 obstacles 56 us with every wave for itself, 39 together).
// Looking at the middle of each gap and then of what that leaves takes fewer
// states but more passes: 72 us.
template <Walk MODE>
__device__ __forceinline__ void wave_edges(const GridWalkArgs &A, int n, int first, int step, BlockEdges &B,
                                           WaveTests &tests)
{
    constexpr bool kSeq = MODE == Walk::kSequence;
    const int lane = lane_id(), half = lane >> 5, s = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WaveEdges &W = B.wave[wave];
    const bool counts = A.m.checked != nullptr;
    int next = first;            // pair
    int head = 0, tail = 0;      // edges: retired, taken
    int looked = 0, listed = 0;  // states
    int from = 1, to = 0;        // indices after the lane's position that are left to list
    bool open = false;           // the last pair's states are being listed
    auto sync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (;;) {
        const bool more = 2 * (int64_t)next < n; // else the waves of the block go on together
        const int enough = more ? 64 : WaveEdges::kStates - 63;
        if (open) { // list states until there are enough, or no more
            // an invalid edge: nothing more, or (in order) what comes before
            const int bad = W.edge[(tail - 2 + half) % WaveEdges::kEdges].bad;
            if (kSeq) to = min(to, bad - 1);
            else if (!counts && bad != INT_MAX) to = -1;
            uint64_t m = wave_ballot(from <= to);
            while (m && listed - looked < enough) {
                if (from <= to)
                    W.state[(listed + __popcll(m & (((uint64_t)1 << lane) - 1))) % WaveEdges::kStates] =
                        (tail - 2 + half) % WaveEdges::kEdges << 24 | from++;
                listed += __popcll(m);
                m = wave_ballot(from <= to);
            }
            if (m == 0) {
                open = false;
                if (s == 0) W.edge[(tail - 2 + half) % WaveEdges::kEdges].end = listed;
            }
            sync();
        }
        if (!open) { // results of the edges that are done
            const int slot = (head + lane) % WaveEdges::kEdges;
            const bool ready = lane < tail - head && W.edge[slot].end <= looked;
            if (ready && W.edge[slot].id >= 0) {
                const int id = W.edge[slot].id, bad = W.edge[slot].bad, nd = W.edge[slot].nd;
                A.m.out[id] = bad == INT_MAX ? 1 : 0;
                if (kSeq) {
                    if (bad != INT_MAX) A.last_t[id] = (double)(min(bad, nd) - 1) / (double)nd;
                } else if (A.m.checked) {
                    A.m.checked[id] = bad == INT_MAX ? nd : bad + 1;
                }
            }
            head += __popcll(wave_ballot(ready));
        }
        const bool pair = more && !open && listed - looked < 64 && tail - head + 2 <= WaveEdges::kEdges;
        int index = 0, position = 0, done = 0;
        bool live;
        WaveEdges::Edge *E;
        if (pair) {
            const int item = 2 * next + half;
            E = &W.edge[(tail + half) % WaveEdges::kEdges];
            if (item < n && s < 2 * kDof)
                E->ab[s] = !kSeq       ? A.m.surv_ab[(int64_t)item * 2 * kDof + s]
                           : s < kDof ? A.m.a[(int64_t)s * A.m.n + item]
                                      : A.m.b[(int64_t)(s - kDof) * A.m.n + item];
            int nd = 1;
            if (kSeq) {
                sync();
                if (item < n) nd = valid_segment_count<kDof>(E->ab, E->ab + kDof, A.m.lvs, A.m.factor);
            } else if (item < n && s == 2 * kDof) {
                nd = A.m.surv_nd[item];
            }
            const bool mine = item < n && nd - 1 <= kLongWalk;
            if (s == 2 * kDof) {
                E->nd = mine ? nd : 1; // a long one's turn comes
                E->id = !mine ? -1 : kSeq ? item : A.m.list[item];
                E->bad = INT_MAX;
                E->end = INT_MAX;
            }
            if (kSeq && item < n && !mine) {
                if (nd > kMaxSegments) { // reported invalid without a walk
                    if (s == 0) A.m.out[item] = 0;
                } else {
                    if (s < 2 * kDof) A.m.surv_ab[(int64_t)item * 2 * kDof + s] = E->ab[s];
                    if (s == 2 * kDof) {
                        A.m.list[item] = item;
                        A.m.surv_nd[item] = nd;
                        list_long(A, item);
                    }
                }
            }
            sync();
            nd = E->nd;
            // in order, or (short edges) all of them; lane 0 of a half: s1 or s2
            position = nd > 32 ? (s ? heap_of_slot(s, 5) : 0) : s;
            live = position > 0 ? position < nd : kSeq ? E->id >= 0 : nd > 32;
            index = live && position > 0 ? bisection_index(position - 1, nd) : 0;
            if (kSeq && position == 0) index = max(nd, 1);
        } else if (more) {
            // (a ring full of edges whose states are all looked at cannot be: they are retired)
            done = min(64, listed - looked);
            live = lane < done;
            const int st = live ? W.state[(looked + lane) % WaveEdges::kStates] : 0;
            E = &W.edge[live ? st >> 24 : head % WaveEdges::kEdges];
            index = st & 0xffffff;
        } else {
            if (lane == 0) {
                B.looked[wave] = looked;
                B.held[wave] = listed - looked;
            }
            __syncthreads();
            // the block's next 256 states, ring after ring
            int at = threadIdx.x, ring = -1, before = 0, st = 0;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const int held = __builtin_amdgcn_readfirstlane(B.held[w]);
                if (w == wave) done = min(max(256 - before, 0), held);
                if (ring < 0 && at < held) ring = w;
                if (ring < 0) at -= held;
                before += held;
            }
            if (before == 0) break; // of all four waves
            live = ring >= 0;
            if (live) st = B.wave[ring].state[(B.looked[ring] + at) % WaveEdges::kStates];
            E = &B.wave[live ? ring : 0].edge[live ? st >> 24 : 0];
            index = st & 0xffffff;
        }
        const int nd = live ? E->nd : 1;
        const bool end = kSeq && index >= nd; // s2 itself
        float q[kDof], steps;
        Speeds sp;
        {
            double a[kDof], b[kDof];
#pragma unroll
            for (int j = 0; j < kDof; ++j) {
                a[j] = E->ab[j];
                b[j] = E->ab[kDof + j];
            }
            interpolate_f32<kDof>(a, b, (double)index / (double)nd, q);
            if (kSeq) {
#pragma unroll
                for (int j = 0; j < kDof; ++j) q[j] = end ? (float)b[j] : q[j];
            }
            sp.far = kFarUnits;
            sp.near = kClearReachUnits;
            if (pair) edge_speeds(a, b, nd, (float)nd * (0.5f / 32.0f) + 1.0f, sp);
        }
        const bool hit = state_hit1<true>(A.g, q, live, tests, sp, &steps);
        if (pair) {
            if (hit && (kSeq || position > 0)) atomicMin(&E->bad, kSeq ? index : position);
            const int k = hit || !live ? 0 : (int)fminf(steps, 65536.0f);
            sync();
            // what neither this position nor the next one reaches
            const int right = __shfl(index - k, s == 31 ? lane - 31 : lane + 1);
            from = kSeq && s == 0 ? 1 : index + k + 1;
            to = !kSeq && s == 31 ? E->nd - 1 : right - 1;
            // all looked at, or invalid: the bisection's first positions come first
            if (E->nd <= 32 || (!kSeq && E->bad != INT_MAX)) to = -1;
            next += step;
            tail += 2;
            open = true;
        } else {
            if (hit) atomicMin(&E->bad, kSeq ? index : 1 + bisection_rank(index, nd));
            looked += done;
            sync();
            if (!more) __syncthreads(); // the others have read this ring
        }
    }
}

// Survivors of the s2 pass: when there are no more than blocks, a block walks
// each to its end; else waves walk pairs of them (an edge that fails does so
// early, and half a wave finds out).  Last, all blocks together walk the long
// ones.
__global__ void __launch_bounds__(256, 4) grid_survivors_kernel(GridWalkArgs A)
{
    __shared__ Rounds R;
    __shared__ WaveTests tests[4];
    __shared__ BlockEdges edges;
    clear_next(A);
    const int n = A.counts[0], n_long = A.counts[1];
    const bool wide = n <= (int)gridDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (!wide) wave_edges<Walk::kBisect>(A, n, blockIdx.x * 4 + wave, gridDim.x * 4, edges, tests[wave]);
    int turn = 0, l = -1;
    Item<Walk::kBisect> I;
    for (int64_t next = wide ? blockIdx.x : n;;) {
        const bool is_long = next >= n;
        int slot = (int)next;
        if (is_long) {
            if (++l >= n_long) break;
            slot = A.long_slot[l];
        }
        next += gridDim.x;
        I.survivor(A.m, slot);
        if (!is_long && I.total - 1 > kLongWalk) continue; // its turn comes (block-uniform)
        const int b = walk_item(A, I, 1 + (is_long ? (int64_t)blockIdx.x * 256 : 0), I.total,
                                is_long ? (int64_t)gridDim.x * 256 : 256, is_long ? &A.long_bad[l] : nullptr, R, turn,
                                tests);
        if (threadIdx.x == 0) { // (no `continue` for the other lanes: they would walk on without this one)
            if (is_long) finish_long(A, I, b, &A.long_bad[l], &A.ticket[l], gridDim.x);
            else I.result(A, b);
        }
    }
}

// Up to kWideItems edges (kBisect with s2 as position 0, kSequence) or lists: a
// block walks each to its end, in one launch with every position in flight at
// once.  The kHelpers blocks after them look through all items for long ones
// (a few loads a thread, while the others walk) and walk those together.
template <Walk MODE>
__global__ void __launch_bounds__(256, 4) grid_wide_kernel(GridWalkArgs A)
{
    __shared__ Rounds R;
    __shared__ WaveTests tests[4];
    __shared__ int longs[kWideItems], n_longs;
    clear_next(A);
    constexpr int from = MODE == Walk::kSequence ? 1 : 0;
    const int n = (int)A.m.n, helper = (int)blockIdx.x - n;
    Item<MODE> I;
    int turn = 0, left = 1;
    if (helper >= 0) {
        if (threadIdx.x == 0) n_longs = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < n; i += 256) {
            if (MODE == Walk::kList) I.list(A, i);
            else I.edge(A.m, i);
            if (!I.nd_too_many() && I.total - from > kLongWalk) longs[atomicAdd(&n_longs, 1)] = i;
        }
        __syncthreads();
        left = n_longs;
    }
    for (; left > 0; --left) { // block-uniform
        const int id = helper < 0 ? (int)blockIdx.x : longs[left - 1];
        if (MODE == Walk::kList) I.list(A, id);
        else I.one_edge(A.m, id);
        const bool none = I.nd_too_many(); // reported invalid without a walk (its s2 is looked at)
        if (helper < 0 && !none && I.total - from > kLongWalk) return;
        const int end = none ? (MODE == Walk::kBisect ? 1 : 0) : I.total;
        const int b = walk_item(A, I, from + (int64_t)max(helper, 0) * 256, end,
                                helper < 0 ? 256 : (int64_t)kHelpers * 256, helper < 0 ? nullptr : &A.wide_bad[id], R,
                                turn, tests);
        if (threadIdx.x == 0) {
            if (none) {
                A.m.out[id] = 0;
                if (A.m.checked) A.m.checked[id] = b == 0 ? 1 : 0;
            } else if (helper < 0) {
                I.result(A, b);
            } else {
                finish_long(A, I, b, &A.wide_bad[id], &A.wide_ticket[id], kHelpers);
            }
        }
    }
}

// More edges in order (kSequence): waves walk pairs of them.
__global__ void __launch_bounds__(256, 4) grid_sequence_kernel(GridWalkArgs A)
{
    __shared__ WaveTests tests[4];
    __shared__ BlockEdges edges;
    clear_next(A);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    wave_edges<Walk::kSequence>(A, (int)A.m.n, blockIdx.x * 4 + wave, gridDim.x * 4, edges, tests[wave]);
}

// More lists: a wave walks the first 64 states of each.
__global__ void __launch_bounds__(256, 4) grid_first_kernel(GridWalkArgs A)
{
    __shared__ WaveTests tests[4];
    clear_next(A);
    const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (id >= A.m.n) return;
    Item<Walk::kList> I;
    I.list(A, id);
    const int slot = (int)id, done = min(I.total, 64);
    const int b = wave_walk(A, I, 0, done, tests);
    if (lane_id() != 0) return;
    bool left = false;
    if (b != INT_MAX || done == I.total) {
        I.result(A, b);
    } else {
        left = I.total - done <= kLongWalk;
        if (!left) list_long(A, slot);
    }
    A.rest[slot] = left;
}

// What the kernel before left: a block per list; then all blocks together the
// long edges or lists.
template <Walk MODE>
__global__ void __launch_bounds__(256, 4) grid_rest_kernel(GridWalkArgs A)
{
    __shared__ Rounds R;
    __shared__ WaveTests tests[4];
    constexpr int from = MODE == Walk::kSequence ? 1 : 64;
    const int n_long = A.counts[1];
    const int64_t n = MODE == Walk::kSequence ? 0 : A.m.n;
    Item<MODE> I;
    const int lane = lane_id();
    // the block's slots are blockIdx.x + i gridDim.x (every wave reads the same
    // 64 flags at a time), then all blocks' long items
    int64_t i0 = -64;
    uint64_t open = 0;
    int turn = 0, l = -1;
    for (;;) {
        int slot = -1;
        if (l < 0) {
            while (open == 0) {
                i0 += 64;
                if (blockIdx.x + i0 * gridDim.x >= n) break;
                const int64_t mine = blockIdx.x + (i0 + lane) * gridDim.x;
                open = wave_ballot(mine < n && A.rest[mine < n ? mine : 0] != 0);
            }
            if (open) {
                slot = (int)(blockIdx.x + (i0 + lowest_bit(open)) * gridDim.x);
                open &= open - 1;
            }
        }
        const bool is_long = slot < 0;
        if (is_long) {
            if (++l >= n_long) break;
            slot = A.long_slot[l];
        }
        if (MODE == Walk::kList) I.list(A, slot);
        else I.survivor(A.m, slot);
        const int b = walk_item(A, I, from + (is_long ? (int64_t)blockIdx.x * 256 : 0), I.total,
                                is_long ? (int64_t)gridDim.x * 256 : 256, is_long ? &A.long_bad[l] : nullptr, R, turn,
                                tests);
        if (threadIdx.x == 0) { // (no `continue` for the other lanes: they would walk on without this one)
            if (is_long) finish_long(A, I, b, &A.long_bad[l], &A.ticket[l], gridDim.x);
            else I.result(A, b);
        }
    }
}

// One edge by value, walked by a block (the per-call path).
__global__ void __launch_bounds__(256, 4) grid_motion_single_kernel(GridView g, Edge1 E, double lvs, unsigned factor,
                                                                    int *result)
{
    __shared__ Rounds R;
    __shared__ WaveTests tests[4];
    GridWalkArgs A{};
    A.g = g;
    Item<Walk::kBisect> I;
#pragma unroll
    for (int j = 0; j < kDof; ++j) {
        I.a[j] = E.a[j];
        I.b[j] = E.b[j];
    }
    I.nd = valid_segment_count<kDof>(I.a, I.b, lvs, factor);
    I.total = max(I.nd, 1);
    int turn = 0;
    int b = 0; // too many segments: invalid
    if (!I.nd_too_many()) b = walk_item(A, I, 0, I.total, 256, nullptr, R, turn, tests);
    if (threadIdx.x == 0) *result = b == INT_MAX ? 1 : 0;
}

// One state by value.
__global__ void __launch_bounds__(64) grid_validate_single_kernel(GridView g, State1 s, int *result)
{
    __shared__ WaveTests tests;
    const int lane = lane_id();
    const uint64_t H = wave_ballot(state_hit8(g, (float)s.q[min(lane & 7, kDof - 1)], lane < 8, tests));
    if (lane == 0) *result = H ? 0 : 1;
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
static unsigned grid_of(int64_t units, int64_t per)
{
    return (unsigned)((units + per - 1) / per);
}

// States (or edges) from which on one lane per state beats eight: 131,072 fill
// every SIMD with two waves of 64 states; below, eight lanes have more in flight.
constexpr int64_t kLaneStates = 131072;
template <typename T>
void launch_grid_validate(const GridView &g, const T *q, int64_t n, uint8_t *out, hipStream_t s)
{
    if (n <= 0) return;
    ProfScope ps("validate_states", s);
    if (n >= kLaneStates)
        hipLaunchKernelGGL((grid_validate_kernel<1, T>), dim3(grid_of(n, 256)), dim3(256), 0, s, g, q, n, out);
    else
        hipLaunchKernelGGL((grid_validate_kernel<8, T>), dim3(grid_of(n, 32)), dim3(256), 0, s, g, q, n, out);
    OA_HIP(hipGetLastError());
}
template void launch_grid_validate<float>(const GridView &, const float *, int64_t, uint8_t *, hipStream_t);
template void launch_grid_validate<double>(const GridView &, const double *, int64_t, uint8_t *, hipStream_t);

static GridWalkArgs walk_args(const GridView &g, const MotionArgs &m, const GridScratch &w)
{
    GridWalkArgs A{};
    A.g = g;
    A.m = m;
    A.m.list = w.list;
    A.m.surv_nd = w.surv_nd;
    A.m.surv_ab = w.surv_ab;
    A.m.list_count = w.counts;
    A.rest = w.rest;
    A.long_slot = w.long_slot;
    A.long_bad = w.long_bad;
    A.ticket = w.ticket;
    A.wide_bad = w.wide;
    A.wide_ticket = w.wide + kWideItems;
    A.counts = w.counts;
    A.next = w.next;
    return A;
}

template <Walk MODE>
static void launch_wide(const GridWalkArgs &A, hipStream_t s)
{
    hipLaunchKernelGGL((grid_wide_kernel<MODE>), dim3((unsigned)A.m.n + kHelpers), dim3(256), 0, s, A);
    OA_HIP(hipGetLastError());
}

// Edges in order or lists.
template <Walk MODE>
static void launch_items(const GridWalkArgs &A, hipStream_t s)
{
    if (A.m.n <= kWideItems) return launch_wide<MODE>(A, s);
    const unsigned blocks = (unsigned)num_cus();
    if (MODE == Walk::kSequence)
        hipLaunchKernelGGL(grid_sequence_kernel, dim3(blocks * 8), dim3(256), 0, s, A);
    else
        hipLaunchKernelGGL(grid_first_kernel, dim3(grid_of(A.m.n, 4)), dim3(256), 0, s, A);
    hipLaunchKernelGGL((grid_rest_kernel<MODE>), dim3(blocks * 4), dim3(256), 0, s, A);
    OA_HIP(hipGetLastError());
}

void launch_motion_single(const GridView &g, const Edge1 &E, double lvs, unsigned factor, int *result, hipStream_t s)
{
    hipLaunchKernelGGL(grid_motion_single_kernel, dim3(1), dim3(256), 0, s, g, E, lvs, factor, result);
    OA_HIP(hipGetLastError());
}

void launch_validate_single(const GridView &g, const State1 &st, int *result, hipStream_t s)
{
    hipLaunchKernelGGL(grid_validate_single_kernel, dim3(1), dim3(64), 0, s, g, st, result);
    OA_HIP(hipGetLastError());
}

static void launch_endpoints(const GridWalkArgs &A, hipStream_t s)
{
    if (A.m.n >= kLaneStates)
        hipLaunchKernelGGL(grid_endpoint1_kernel, dim3(grid_of(A.m.n, 256)), dim3(256), 0, s, A);
    else
        hipLaunchKernelGGL(grid_endpoint8_kernel, dim3(grid_of(A.m.n, 32)), dim3(256), 0, s, A);
    OA_HIP(hipGetLastError());
}

static void launch_survivors(const GridWalkArgs &A, hipStream_t s)
{
    hipLaunchKernelGGL(grid_survivors_kernel, dim3((unsigned)num_cus() * 8), dim3(256), 0, s, A);
    OA_HIP(hipGetLastError());
}

void launch_grid_motions(const GridView &g, const MotionArgs &m, const GridScratch &w, bool fused, hipStream_t s)
{
    if (m.n <= 0) return;
    const GridWalkArgs A = walk_args(g, m, w);
    if (m.n <= kWideItems) {
        ProfScope ps(fused ? "motion_fused" : "motion_walk", s);
        launch_wide<Walk::kBisect>(A, s);
        return;
    }
    if (fused) {
        ProfScope ps("motion_fused", s);
        launch_endpoints(A, s);
        launch_survivors(A, s);
        return;
    }
    {
        ProfScope ps("motion_endpoint", s);
        launch_endpoints(A, s);
    }
    ProfScope ps("motion_chunk", s);
    launch_survivors(A, s);
}

void launch_grid_last_valid(const GridView &g, const MotionArgs &m, double *last_t, const GridScratch &w,
                            hipStream_t s)
{
    if (m.n <= 0) return;
    GridWalkArgs A = walk_args(g, m, w);
    A.last_t = last_t;
    ProfScope ps("motion_last_valid", s);
    launch_items<Walk::kSequence>(A, s);
}

void launch_grid_state_lists(const GridView &g, const double *q_soa, int64_t n_states, const int64_t *offsets,
                             int64_t n_lists, uint8_t *out, int32_t *first_invalid, const GridScratch &w,
                             hipStream_t s)
{
    if (n_lists <= 0) return;
    MotionArgs m{};
    m.n = n_lists;
    m.out = out;
    m.checked = first_invalid;
    GridWalkArgs A = walk_args(g, m, w);
    A.q = q_soa;
    A.n_states = n_states;
    A.offsets = offsets;
    ProfScope ps("state_lists", s);
    launch_items<Walk::kList>(A, s);
}

} // namespace ompl_amd
