// Spatial index of the nearest-neighbour structure (nn_tree.hpp).
//
// Build: the points are put into one order whose consecutive runs are compact,
// and cut into tiles of 64.  Every dimension but the last is cut into cells of
// equal counts (quantiles, from a sample); the cells, walked in reflected
// (boustrophedon) order, are columns along the last dimension, and a column's
// points are sorted by it, upwards and downwards in turn.  Consecutive points
// are then neighbours also where a column ends.  A column is dealt to buckets
// of at most a thousand points or so by counting, and one workgroup sorts each bucket
// in LDS: 100,000 points in 7 dimensions take 9 launches, where one radix sort
// per dimension (nested cuts) took about 70 and 440 us; a CPU model gives 40.8
// tiles per 10-NN query for this order and 38.7 for the nested one (SE3 1M:
// 32.4 and 39.8).
//
// Search: one wave per query (or W waves, for batches too small to fill the
// device).  Lane l of the wave tests child l of a node (64 boxes at once) or
// point l of a tile, children are taken nearest box first, and the query's 64
// best keys sit one per lane in ascending order.  A box is skipped when its
// squared distance, evaluated in the operation order of the exact distance, is
// above the k-th key's: rounding is monotone, so no point of a skipped box has
// an exact distance at or below it, and the lists are those of the full scan.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <climits>

#include "arm_device.hpp"
#include "common.hpp"
#include "nn_device.hpp"
#include "nn_tree.hpp"

namespace ompl_amd {

// ---------------------------------------------------------------------------
// build
// ---------------------------------------------------------------------------
constexpr int kSample = 2048;       // values per dimension that the cuts are made from,
constexpr int kSmallSample = 1024;  // and below kSmallPoints, whose cells are fewer (2 us less)
constexpr int64_t kSmallPoints = 16384;
static_assert(kSample <= kTreeMinPoints, "a point for every run");
constexpr int kKnots = 512;         // most quantiles of a dimension that are looked up; finer cuts interpolate
constexpr int kBins = 512;          // cells per dimension of the queries' search order
constexpr int kBucketPoints = 768;  // points a bucket is meant to hold: the cuts vary with the sample, and a sort of more
                                    // than 1,024 pads to 2,048 (SE3 1M: sorts 48 us, 63 with 1,024 meant)
constexpr int kBucketSort = 4096;   // points sorted at once; a fuller bucket (many equal coordinates) in parts

// A build's cuts.  They come from a sample of each coordinate, not from its
// extent: one far point, or a heavy tail, would leave all others in one cell of
// equal widths, thus in one bucket (adding 1,000,000 points 32 ms in place of 0.4).
struct TreePlan {
    int cuts[8];              // cells per dimension; the last dimension's: buckets per column
    int finite[8];            // finite values of the sample
    float base[8], scale[8];  // cell of a query = (x - base) * scale
    float sample[8][kSample]; // ascending
};

__device__ __forceinline__ float from_ordered(uint32_t u)
{
    return __uint_as_float(u & 0x80000000u ? u ^ 0x80000000u : ~u);
}

// One round of a bitonic sort of the block's values, four a thread (value e of
// thread t is number 4 t + e): exchanges with number ^ J, ascending where K is clear.
template <int K, int J>
__device__ __forceinline__ void sample_round(uint32_t v[4], uint32_t *key)
{
    const int i0 = 4 * threadIdx.x;
    uint32_t o[4];
    if constexpr (J >= 256) {
        *reinterpret_cast<uint4 *>(&key[i0]) = make_uint4(v[0], v[1], v[2], v[3]);
        __syncthreads();
        const uint4 w = *reinterpret_cast<const uint4 *>(&key[i0 ^ J]);
        o[0] = w.x, o[1] = w.y, o[2] = w.z, o[3] = w.w;
        __syncthreads();
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = J >= 4 ? (uint32_t)__shfl_xor((int)v[e], J / 4) : v[e ^ (J & 3)];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int i = i0 + e;
        v[e] = ((i & J) == 0) == ((i & K) == 0) ? min(v[e], o[e]) : max(v[e], o[e]);
    }
    if constexpr (J > 1) sample_round<K, J / 2>(v, key);
}

template <int K>
__device__ __forceinline__ void sample_sort(uint32_t v[4], uint32_t *key)
{
    if constexpr (K > 2) sample_sort<K / 2>(v, key);
    sample_round<K, K / 2>(v, key);
}

// The sorted sample of dimension blockIdx.x: a point at random (by a hash) of
// each of SAMPLE equal runs, so that no regular order of the points shows.
// Exchanges within a wave are shuffles: 6 of the sort's 66 rounds (2,048 values)
// wait for other waves.
template <int SAMPLE>
__global__ void __launch_bounds__(SAMPLE / 4) tree_sample_kernel(const float *__restrict__ pts, int64_t n, int dim,
                                                                 TreePlan *__restrict__ plan)
{
    __shared__ uint32_t key[SAMPLE];
    __shared__ int waves_finite[SAMPLE / 256];
    const int d = blockIdx.x, i0 = 4 * threadIdx.x;
    uint32_t v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t from = n * (i0 + e) / SAMPLE, to = n * (i0 + e + 1) / SAMPLE;
        const uint32_t skip = __umulhi((uint32_t)(i0 + e) * 2654435761u, (uint32_t)(to - from));
        const float x = pts[(from + skip) * dim + d];
        v[e] = fabsf(x) < 3e38f ? ordered_bits(x) : ~0u; // not finite: last
    }
    sample_sort<SAMPLE>(v, key);
    int finite = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        plan->sample[d][i0 + e] = from_ordered(v[e]);
        finite += __popcll(__ballot(v[e] != ~0u));
    }
    if ((threadIdx.x & 63) == 0) waves_finite[threadIdx.x >> 6] = finite;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SAMPLE / 256; ++w) finite += waves_finite[w];
        plan->finite[d] = finite;
    }
}

// Chooses the cuts (one block), and clears the bucket counts.  The dimension
// whose cells are longest gets one cut more until there are as many cells as
// tiles; the last dimension is then cut into buckets instead.  A dimension's
// length is that of its sample without the ends' 64ths (nothing for one that is
// nearly constant, whatever its few other values).
__global__ void __launch_bounds__(256) plan_kernel(int64_t n, int tdim, TreePlan *__restrict__ plan,
                                                   uint32_t *__restrict__ counts, int64_t buckets)
{
    for (int64_t i = threadIdx.x; i < buckets; i += blockDim.x) counts[i] = 0;
    if (threadIdx.x >= 64) return;
    // lane j holds dimension j
    const int j = threadIdx.x;
    float lo = 0.0f, ext = 0.0f;
    auto length = [&](int from, int to) {
        lo = plan->sample[j][from];
        ext = plan->sample[j][to] - lo;
        if (!(ext > 0.0f && ext < 3e38f)) ext = 0.0f;
    };
    const int m = j < tdim ? plan->finite[j] : 0;
    if (m > 0) length(m / 64, m - 1 - m / 64);
    if (__ballot(ext > 0.0f) == 0 && m > 0) length(0, m - 1); // nearly all points equal
    if (j < tdim) {
        plan->base[j] = lo;
        plan->scale[j] = ext > 0.0f ? (float)kBins / ext : 0.0f;
    }
    const int64_t tiles = (n + kTile - 1) / kTile;
    int cuts = 1;
    int64_t cells = 1;
    while (cells < tiles) {
        float longest = j < tdim ? ext / (float)cuts : -1.0f;
        const float mine = longest;
#pragma unroll
        for (int d = 1; d < 8; d <<= 1) longest = fmaxf(longest, __shfl_xor(longest, d));
        longest = __shfl(longest, 0);
        if (!(longest > 0.0f)) break; // all points equal
        const int best = __builtin_ctzll(__ballot(mine == longest));
        const int64_t c = __shfl(cuts, best);
        // a long thin extent gets its cuts in steps of an eighth
        const int64_t more = c / 8 + 1;
        if (j == best) cuts += (int)more;
        cells = cells / c * (c + more);
    }
    int64_t columns = 1;
    for (int d = 0; d + 1 < tdim; ++d) columns *= __shfl(cuts, d);
    if (j == tdim - 1) cuts = (int)max((int64_t)1, (n + columns * kBucketPoints - 1) / (columns * kBucketPoints));
    if (j < tdim) plan->cuts[j] = cuts;
}

// Most buckets plan_kernel can ask for: its cells overshoot the tile count by
// at most a factor of two (one cut more of one), and a column has at most one
// bucket more than its points need.
static int64_t max_buckets(int64_t n)
{
    return 2 * ((n + kTile - 1) / kTile) + (n + kBucketPoints - 1) / kBucketPoints + 64;
}

__device__ __forceinline__ float bin_of(const TreePlan &plan, int j, float x)
{
    return fminf(fmaxf((x - plan.base[j]) * plan.scale[j], 0.0f), (float)kBins - 0.001f); // NaN: 0
}

// Each point's bucket and its arrival number there.
__global__ void __launch_bounds__(1024) tree_buckets_kernel(const float *__restrict__ pts, int64_t n, int dim,
                                                            int tdim, const TreePlan *__restrict__ plan,
                                                            uint32_t *__restrict__ counts, uint2 *__restrict__ place)
{
    __shared__ float knot[kTreeDimMax][kKnots + 1]; // ascending; [0] and [knots]: the sample's ends
    const int lane = threadIdx.x & 63;
    for (int j = 0; j < tdim; ++j) {
        const int knots = min(plan->cuts[j], kKnots), m = plan->finite[j];
        for (int i = threadIdx.x; i <= knots; i += blockDim.x)
            knot[j][i] = m > 0 ? plan->sample[j][min((int)((int64_t)i * m / knots), m - 1)] : 0.0f;
    }
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        uint32_t idx = 0;
        float coord[kTreeDimMax]; // read together
#pragma unroll
        for (int j = 0; j < kTreeDimMax; ++j)
            if (j < tdim) coord[j] = pts[i * dim + j];
#pragma unroll
        for (int j = 0; j < kTreeDimMax; ++j) {
            if (j >= tdim) break;
            const int c = plan->cuts[j], knots = min(c, kKnots);
            int cell = 0;
            if (c > 1) {
                const float x = coord[j];
                // the last knot at or below x (below the second, or not a number: 0)
                for (int step = 1 << (31 - __builtin_clz(knots)); step > 0; step >>= 1)
                    if (cell + step < knots && x >= knot[j][cell + step]) cell += step;
                if (c > knots) {
                    const float lo = knot[j][cell], wide = knot[j][cell + 1] - lo;
                    const float part = wide > 0.0f ? fminf(fmaxf((x - lo) / wide, 0.0f), 1.0f) : 0.0f;
                    cell = min(c - 1, (int)(((float)cell + part) * ((float)c / (float)knots)));
                }
            }
            // reflected order: every other run of a dimension's cells is walked backwards
            idx = idx * (uint32_t)c + (uint32_t)((idx & 1) ? c - 1 - cell : cell);
        }
        // one atomic for lanes of the same bucket (the first four such groups):
        // points of equal coordinates would queue up at one address
        int lead = lane, before = 0, group = 1;
        bool open = true;
        for (int r = 0; r < 4; ++r) {
            const uint64_t m = __ballot(open);
            if (m == 0) break;
            const int l = __builtin_ctzll(m);
            const bool same = open && idx == (uint32_t)__builtin_amdgcn_readlane((int)idx, l);
            const uint64_t g = __ballot(same);
            if (same) {
                lead = l;
                before = __popcll(g & (((uint64_t)1 << lane) - 1));
                group = __popcll(g);
                open = false;
            }
        }
        uint32_t at = 0;
        if (lead == lane) at = atomicAdd(&counts[idx], (uint32_t)group);
        place[i] = make_uint2(idx, (uint32_t)__shfl((int)at, lead) + (uint32_t)before);
    }
}

// counts[i] becomes the first place of bucket i, counts[buckets] the total (one block).
__global__ void __launch_bounds__(1024) tree_scan_kernel(uint32_t *__restrict__ counts, int64_t buckets)
{
    __shared__ uint32_t part[16];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t carry = 0;
    for (int64_t base = 0; base < buckets; base += 4096) {
        uint32_t v[4], sum = 0;
        const int64_t at = base + 4 * (int64_t)threadIdx.x;
#pragma unroll
        for (int i = 0; i < 4; ++i) sum += v[i] = at + i < buckets ? counts[at + i] : 0;
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)incl, d);
            if (lane >= d) incl += u;
        }
        if (lane == 63) part[w] = incl;
        __syncthreads();
        uint32_t before = carry, all = 0;
        for (int i = 0; i < 16; ++i) {
            if (i < w) before += part[i];
            all += part[i];
        }
        uint32_t run = before + incl - sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (at + i < buckets) counts[at + i] = run;
            run += v[i];
        }
        carry += all;
        __syncthreads();
    }
    if (threadIdx.x == 0) counts[buckets] = carry;
}

// (last coordinate, id) of every point at its bucket's place.
__global__ void __launch_bounds__(256) tree_scatter_kernel(const float *__restrict__ pts, int64_t n, int dim, int tdim,
                                                           const uint32_t *__restrict__ first,
                                                           const uint2 *__restrict__ place,
                                                           unsigned long long *__restrict__ keys)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint2 p = place[i];
    keys[first[p.x] + p.y] = ((unsigned long long)ordered_bits(pts[i * dim + tdim - 1]) << 32) | (uint32_t)i;
}

// Sorts the buckets by the last coordinate, each in the direction of its column:
// block b the first kBucketSort points of bucket b; the blocks after those each
// the part that starts in a run of kBucketSort places, if any, of the bucket that
// holds the run's first place (the parts of a bucket start kBucketSort apart, so
// a run has one at most).
__global__ void __launch_bounds__(256) tree_sort_kernel(const TreePlan *__restrict__ plan, int tdim, int64_t buckets,
                                                        const uint32_t *__restrict__ first,
                                                        const unsigned long long *__restrict__ keys,
                                                        uint32_t *__restrict__ perm)
{
    __shared__ unsigned long long buf[kBucketSort];
    int64_t b = blockIdx.x;
    uint32_t at;
    if (b < buckets) {
        at = first[b];
    } else {
        const uint32_t run = (uint32_t)(b - buckets) * kBucketSort;
        if (run >= first[buckets]) return;
        int64_t lo = 0, hi = buckets; // first[lo] <= run < first[hi]
        while (hi - lo > 1) {
            const int64_t mid = (lo + hi) / 2;
            if (first[mid] <= run) lo = mid;
            else hi = mid;
        }
        b = lo;
        const uint32_t part = (run - first[b] + kBucketSort - 1) / kBucketSort;
        if (part == 0) return; // block b's
        at = first[b] + part * kBucketSort;
    }
    const uint32_t end = first[b + 1];
    if (at >= end) return; // block-uniform
    const bool down = ((b / plan->cuts[tdim - 1]) & 1) != 0;
    const int m = (int)min((uint32_t)kBucketSort, end - at);
    int np2 = 1;
    while (np2 < m) np2 <<= 1;
    for (int i = threadIdx.x; i < np2; i += blockDim.x) {
        const unsigned long long k = i < m ? keys[at + i] : ~0ull;
        buf[i] = down && i < m ? k ^ 0xffffffff00000000ull : k;
    }
    __syncthreads();
    for (int k = 2; k <= np2; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int p = threadIdx.x; p < np2 / 2; p += blockDim.x) {
                const int i = 2 * p - (p & (j - 1)), o = i + j;
                const unsigned long long x = buf[i], y = buf[o];
                if ((x > y) == ((i & k) == 0)) {
                    buf[i] = y;
                    buf[o] = x;
                }
            }
            __syncthreads();
        }
    for (int i = threadIdx.x; i < m; i += blockDim.x) perm[at + i] = (uint32_t)buf[i];
}

__device__ __forceinline__ uint32_t spread_bits(uint32_t v, int dims)
{
    uint32_t r = 0;
    for (int b = 0; b < 10; ++b) r |= ((v >> b) & 1u) << (b * dims);
    return r;
}

// Writes the tiles (one wave each) and their boxes.
__global__ void __launch_bounds__(256) tree_gather_kernel(const float *__restrict__ pts,
                                                          const uint8_t *__restrict__ removed, int64_t n, int dim,
                                                          int tdim, int64_t tiles, const uint32_t *__restrict__ perm,
                                                          NNTree T, uint32_t *__restrict__ live)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *live = (uint32_t)n;
    const int lane = threadIdx.x & 63;
    const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (t >= tiles) return;
    const int64_t src = t * kTile + lane;
    const int64_t id = src < n ? (int64_t)perm[src] : -1;
    const bool there = id >= 0 && !removed[id >= 0 ? id : 0];
    T.sid[t * kTile + lane] = there ? (int32_t)id : -1;
    if (id >= 0) T.pos[id] = (int32_t)(t * kTile + lane);
    for (int j = 0; j < dim; ++j) {
        const float v = id >= 0 ? pts[id * dim + j] : 0.0f;
        T.sp[(t * dim + j) * kTile + lane] = v;
        if (j < tdim) {
            float lo = there ? v : INFINITY, hi = there ? v : -INFINITY;
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) {
                lo = fminf(lo, __shfl_xor(lo, d));
                hi = fmaxf(hi, __shfl_xor(hi, d));
            }
            if (lane == 0) {
                float *b = T.b0 + (t >> 6) * (2 * tdim * kTile) + (t & 63);
                b[j * kTile] = lo;
                b[(tdim + j) * kTile] = hi;
            }
        }
    }
}

// Boxes of `count` parents over `children` child boxes, one wave per parent.
__global__ void __launch_bounds__(256) tree_boxes_kernel(const float *__restrict__ child, int64_t children,
                                                         float *__restrict__ parent, int64_t count, int tdim)
{
    const int lane = threadIdx.x & 63;
    const int64_t p = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (p >= count) return;
    const bool there = p * kTile + lane < children;
    const float *c = child + p * (2 * tdim * kTile) + lane;
    float *o = parent + (p >> 6) * (2 * tdim * kTile) + (p & 63);
    for (int j = 0; j < tdim; ++j) {
        float lo = there ? c[j * kTile] : INFINITY, hi = there ? c[(tdim + j) * kTile] : -INFINITY;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            lo = fminf(lo, __shfl_xor(lo, d));
            hi = fmaxf(hi, __shfl_xor(hi, d));
        }
        if (lane == 0) {
            o[j * kTile] = lo;
            o[(tdim + j) * kTile] = hi;
        }
    }
}

// Search order of a batch: Morton order of the queries' cells, `bits` per dimension.
__global__ void __launch_bounds__(256) query_keys_kernel(const TreePlan *__restrict__ plan, int bits,
                                                         const float *__restrict__ q, int64_t nq, int dim, int tdim,
                                                         uint32_t *__restrict__ keys, uint32_t *__restrict__ vals)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nq) return;
    uint32_t key = 0;
    for (int j = 0; j < tdim; ++j) {
        const uint32_t c = (uint32_t)bin_of(*plan, j, q[i * dim + j]) >> (9 - bits); // 512 bins
        key |= spread_bits(c, tdim) << j;
    }
    keys[i] = key;
    vals[i] = (uint32_t)i;
}

__global__ void tree_remove_kernel(const int32_t *__restrict__ pos, int32_t *__restrict__ sid, int64_t id)
{
    if (threadIdx.x == 0) sid[pos[id]] = -1;
}

// ---------------------------------------------------------------------------
// search
// ---------------------------------------------------------------------------
using u64 = unsigned long long;

__device__ __forceinline__ u64 join_u64(uint32_t lo, uint32_t hi)
{
    return ((u64)hi << 32) | lo;
}

__device__ __forceinline__ u64 lane_u64(u64 v, int j)
{
    return join_u64((uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, j),
                    (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), j));
}

__device__ __forceinline__ u64 shfl_u64(u64 v, int src)
{
    return join_u64((uint32_t)__shfl((int)(uint32_t)v, src), (uint32_t)__shfl((int)(uint32_t)(v >> 32), src));
}

// The previous lane's value; lane 0 gets 0.
__device__ __forceinline__ u64 from_previous_lane(u64 v)
{
    constexpr int kWaveShr1 = 0x138;
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, kWaveShr1, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), kWaveShr1, 0xf, 0xf, true);
    return join_u64((uint32_t)lo, (uint32_t)hi);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_min(uint32_t v)
{
    // lanes without a source take ~0, so the move folds into the minimum
    return min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, CTRL, 0xf, 0xf, false));
}

// Smallest of the lanes' values, wave-uniform.
__device__ __forceinline__ uint32_t wave_min(uint32_t v)
{
    v = dpp_min<0x111>(v); // row_shr 1, 2, 4, 8: the row's minimum in its last lane
    v = dpp_min<0x112>(v);
    v = dpp_min<0x114>(v);
    v = dpp_min<0x118>(v);
    v = dpp_min<0x142>(v); // row_bcast 15, 31: the wave's in lane 63
    v = dpp_min<0x143>(v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Ascending order of the keys of each run of N lanes.
template <int N>
__device__ __forceinline__ u64 wave_sort(u64 v, int lane)
{
#pragma unroll
    for (int k = 2; k <= N; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            const u64 o = shfl_u64(v, lane ^ j);
            const bool keep_min = ((lane & j) == 0) == (k == N || (lane & k) == 0);
            v = (o < v) == keep_min ? o : v;
        }
    return v;
}

// The 64 smallest of two ascending lists, ascending.
__device__ __forceinline__ u64 wave_merge(u64 a, u64 b, int lane)
{
    const u64 r = shfl_u64(b, 63 - lane);
    u64 v = a < r ? a : r; // bitonic
#pragma unroll
    for (int j = 32; j > 0; j >>= 1) {
        const u64 o = shfl_u64(v, lane ^ j);
        v = (o < v) == ((lane & j) == 0) ? o : v;
    }
    return v;
}

template <int METRIC, int DIM>
struct TreeQuery {
    static constexpr int TD = METRIC == OMPL_AMD_METRIC_L2 ? DIM : 3;
    float q[DIM];
    __device__ __forceinline__ void load(const float *__restrict__ src)
    {
#pragma unroll
        for (int j = 0; j < DIM; ++j) q[j] = src[j];
    }
    // Squared distance to child `lane`'s box; the operations of the exact
    // distance on the gap, so never above that of a point inside.
    __device__ __forceinline__ float box2(const float *__restrict__ boxes, int lane) const
    {
        float lo[TD], hi[TD];
#pragma unroll
        for (int j = 0; j < TD; ++j) {
            lo[j] = boxes[j * kTile + lane];
            hi[j] = boxes[(TD + j) * kTile + lane];
        }
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < TD; ++j) {
            const float g = fmaxf(fmaxf(lo[j] - q[j], q[j] - hi[j]), 0.0f);
            s += g * g;
        }
        return s;
    }
    // Squared distance of the coordinates the boxes bound.
    __device__ __forceinline__ float near2(const float e[DIM]) const
    {
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < TD; ++j) {
            const float diff = e[j] - q[j];
            s += diff * diff;
        }
        return s;
    }
    // SE3: |q_e . q_q|
    __device__ __forceinline__ float turn(const float e[DIM]) const
    {
        return fabsf(((e[3] * q[3] + e[4] * q[4]) + e[5] * q[5]) + e[6] * q[6]);
    }
    // The exact distance, from near2's result.
    __device__ __forceinline__ float finish(const float e[DIM], float s) const
    {
        if (METRIC == OMPL_AMD_METRIC_L2) return __builtin_sqrtf(s);
        return exact_dist<METRIC, DIM>(e, q);
    }
};

// One tile's points: lane l's coordinates and id.
template <int DIM>
struct TilePoints {
    float e[DIM];
    int32_t id;
    __device__ __forceinline__ void load(const TreeView &t, int64_t tile, int lane)
    {
        const float *p = t.sp + tile * (DIM * kTile) + lane;
#pragma unroll
        for (int j = 0; j < DIM; ++j) e[j] = p[j * kTile];
        id = t.sid[tile * kTile + lane];
    }
    __device__ __forceinline__ void load_tail(const TreeView &t, int64_t first, int lane)
    {
        const int64_t p = first + lane;
        const bool in = p < t.n;
        const int64_t at = in ? p : t.n - 1;
#pragma unroll
        for (int j = 0; j < DIM; ++j) e[j] = t.pts[at * DIM + j];
        id = in && !t.removed[at] ? (int32_t)p : -1;
    }
};

// Squared bound of a distance bound, widened past the rounding of its square.
__device__ __forceinline__ float bound2(float kd)
{
    return kd * kd * (1.0f + 8e-6f) + 1e-37f;
}

// A query's 64 best keys, one per lane in ascending order, and its bound.
template <int METRIC, int DIM, int W>
struct TreeList {
    u64 key, bkey; // bkey: a key that k points are at or below (wave-uniform)
    float bd, thr; // its distance (infinite while there is none) and squared bound
    u64 *shared;   // W > 1: the smallest bound of the query's waves
    __device__ __forceinline__ void init(u64 *s)
    {
        key = bkey = ~0ull;
        bd = thr = INFINITY;
        shared = s;
    }
    __device__ __forceinline__ void take_bound(u64 b)
    {
        if (b < bkey) {
            bkey = b;
            bd = __uint_as_float((uint32_t)(b >> 32));
            thr = bound2(bd);
        }
    }
    // Adds the lanes' points (CAPTURED: of ids below n); the bound follows.
    template <bool CAPTURED>
    __device__ __forceinline__ void add(const TreeQuery<METRIC, DIM> &Q, const TilePoints<DIM> &P, uint32_t n, int k,
                                        int lane)
    {
        if (W > 1) {
            const u64 b = __hip_atomic_load(shared, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            take_bound(lane_u64(b, 0));
        }
        const float s = Q.near2(P.e);
        bool c = (CAPTURED ? (uint32_t)P.id < n : P.id >= 0) && s <= thr; // false for NaN
        if (METRIC == OMPL_AMD_METRIC_SE3) {
            // the cheap bound first: d^2 >= d_t^2 + d_r^2, d_r^2 >= 2 (1 - |q.x|)
            // (widened past the rounding of the product and of the arc cosine);
            // it leaves no candidate in most of the tiles
            const float dq = Q.turn(P.e);
            c = c && !(s + 2.0f * (1.0f - dq) > thr * (1.0f + 1e-5f) + 4e-6f);
            if (__ballot(c) == 0) return;
            c = c && !certainly_above<METRIC, DIM>(P.e, Q.q, bd);
        }
        if (__ballot(c) == 0) return;
        const float d = Q.finish(P.e, s);
        const u64 nk = c && d == d ? pack_key(d, P.id) : ~0ull;
        u64 m = __ballot(nk < bkey);
        if (m == 0) return;
        if (__popcll(m) > 20) {
            // as many insertions as the sort of a whole tile costs (21 exchanges)
            key = wave_merge(key, wave_sort<64>(nk < bkey ? nk : ~0ull, lane), lane);
        } else {
            do {
                const int j = __builtin_ctzll(m);
                m &= m - 1;
                const u64 v = lane_u64(nk, j);
                // slot s of the new list is max(old[s - 1], min(old[s], v))
                const u64 up = from_previous_lane(key);
                const u64 lo = key < v ? key : v;
                key = up > lo ? up : lo;
            } while (m);
        }
        const u64 kth = lane_u64(key, k - 1);
        if (kth < bkey) {
            take_bound(kth);
            if (W > 1 && lane == 0) atomicMin(shared, kth);
        }
    }
};

// k nearest: W waves per query; with W = 1 a block holds four queries.
// Bound by VALU instructions (62% of the time) and reads past the L2 (7.3 TB/s)
// in large batches (SE3 1M x 65,536, k = 16: 578 us against the full scan's 19,700; about 33 tiles and 8 nodes per query, 100
// instructions a tile and 12 an insertion), by the longest query's read chain
// in small ones (100,000 x 4,096, k = 10, R^7: 71 us against 247).
// CAPTURED: the number of indexed points is read from TreeView::live, and ids
// beyond the view's are left out (a kernel of its own: tests for it in the eager
// one cost 1 to 1.5% of the small batches).
template <int METRIC, int DIM, int W, bool CAPTURED>
__global__ void __launch_bounds__(W == 1 ? 256 : 64 * W) tree_knn_kernel(TreeKnnArgs A)
{
    constexpr int TD = TreeQuery<METRIC, DIM>::TD;
    constexpr int NODE = 2 * TD * kTile;
    __shared__ u64 lists[W > 1 ? W / 2 : 1][kTile];
    __shared__ u64 shared_bound;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t at = xcd_block(blockIdx.x, gridDim.x) * (W == 1 ? 4 : 1) + (W == 1 ? wv : 0);
    const int w = W == 1 ? 0 : wv;
    if (at >= A.nq) return; // W > 1: the grid is the query count
    const int64_t qi = at;
    int k = A.k;
    if (A.kq) {
        const int v = A.kq[qi];
        k = v < 0 ? 0 : (v > A.k ? A.k : v);
    }
    if (k == 0) return; // block-uniform where the block has barriers
    if (W > 1) {
        if (threadIdx.x == 0) shared_bound = ~0ull;
        __syncthreads();
    }
    TreeQuery<METRIC, DIM> Q;
    Q.load(A.q + qi * DIM);
    const TreeView &t = A.t;
    TreeList<METRIC, DIM, W> L;
    L.init(&shared_bound);
    const int64_t in_index = CAPTURED ? (int64_t)*t.live : t.m;
    const uint32_t ids = (uint32_t)t.n;
    // the points added since the index was built
    for (int64_t p = in_index + w * kTile; p < t.n; p += W * kTile) {
        TilePoints<DIM> P;
        P.load_tail(t, p, lane);
        L.template add<CAPTURED>(Q, P, ids, k, lane);
    }
    const int64_t tiles = (in_index + kTile - 1) / kTile, nodes = (tiles + kTile - 1) / kTile,
                  supers = (nodes + kTile - 1) / kTile;
    // Picks the remaining child with the nearest box, or -1 when none is
    // within the bound; lb holds the lanes' squared distances as bits.
    auto pick = [&](u64 &open, uint32_t lb) -> int {
        if (open == 0) return -1;
        const uint32_t best = wave_min((open >> lane) & 1 ? lb : ~0u);
        if (!(__uint_as_float(best) <= L.thr)) return -1;
        const int j = __builtin_ctzll(open & __ballot(lb == best));
        open &= ~((u64)1 << j);
        return j;
    };
    auto first = [](int64_t count) -> u64 { return count >= 64 ? ~0ull : ((u64)1 << count) - 1; };
    auto boxes = [&](const float *b, int64_t count) -> uint32_t {
        return __float_as_uint(lane < count ? Q.box2(b, lane) : INFINITY);
    };
    // W waves share a node's tiles
    u64 mine = ~0ull;
    if (W > 1) {
        mine = 0;
        for (int i = w; i < 64; i += W) mine |= (u64)1 << i;
    }
    for (int64_t s0 = 0; s0 < supers; s0 += 64) {
        u64 open2 = first(supers - s0);
        const uint32_t lb2 = supers == 1 ? 0u : boxes(t.b2 + (s0 >> 6) * NODE, supers - s0);
        for (int a; (a = pick(open2, lb2)) >= 0;) {
            const int64_t sn = s0 + a, n0 = sn * kTile;
            u64 open1 = first(nodes - n0);
            const uint32_t lb1 = nodes == 1 ? 0u : boxes(t.b1 + sn * NODE, nodes - n0);
            for (int b; (b = pick(open1, lb1)) >= 0;) {
                const int64_t node = n0 + b, t0 = node * kTile;
                u64 open0 = first(tiles - t0) & mine;
                const uint32_t lb0 = boxes(t.b0 + node * NODE, tiles - t0);
                // the next tile's points are in flight while one is added
                TilePoints<DIM> P[2];
                int c = pick(open0, lb0);
                if (c < 0) continue;
                P[0].load(t, t0 + c, lane);
                for (;;) {
                    const int nx = pick(open0, lb0);
                    if (nx >= 0) P[1].load(t, t0 + nx, lane);
                    L.template add<CAPTURED>(Q, P[0], ids, k, lane);
                    if (nx < 0) break;
                    P[0] = P[1];
                }
            }
        }
    }
    u64 key = L.key;
    if (W > 1) {
        // halves of the waves hand their lists to the other half
#pragma unroll
        for (int h = W / 2; h > 0; h >>= 1) {
            __syncthreads();
            if (w >= h && w < 2 * h) lists[w - h][lane] = key;
            __syncthreads();
            if (w < h) key = wave_merge(key, lists[w][lane], lane);
        }
        if (w != 0) return;
    }
    const int64_t base = A.out_off ? A.out_off[qi] : qi * A.k;
    if (lane < k) {
        A.out_d[base + lane] = key == ~0ull ? INFINITY : __uint_as_float((uint32_t)(key >> 32));
        A.out_i[base + lane] = key == ~0ull ? -1 : (int32_t)(uint32_t)key;
    }
}

// All points within the radius: one wave per query, a block holds four.
// Bound by VALU instructions once the queries are in space order (SE3 1M x 65,536,
// r = 0.98: 190 us of a 245 us call, 86% of it issuing them, 98% L2 hits; without
// the order by reads, 430 us; the full scan took 11,862).
template <int METRIC, int DIM>
__global__ void __launch_bounds__(256) tree_radius_kernel(TreeRadiusArgs A)
{
    __shared__ u64 kept[4][kTile]; // a slot's keys, until they are sorted
    constexpr int TD = TreeQuery<METRIC, DIM>::TD;
    constexpr int NODE = 2 * TD * kTile;
    const int lane = threadIdx.x & 63;
    const int64_t at = xcd_block(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (at >= A.nq) return;
    const int64_t qi = A.order ? A.order[at] : at;
    const float r = A.rq ? A.rq[qi] : A.radius;
    const TreeView &t = A.t;
    int64_t found = 0;
    u64 *mine = kept[threadIdx.x >> 6];
    if (r >= 0.0f) { // else (negative or not a number) no results
        TreeQuery<METRIC, DIM> Q;
        Q.load(A.q + qi * DIM);
        const float thr = bound2(r);
        uint64_t *out = A.offsets ? A.keys + A.offsets[qi] : nullptr;
        const int64_t room = A.offsets ? A.offsets[qi + 1] - A.offsets[qi] : A.slot_cap;
        auto add = [&](const TilePoints<DIM> &P) {
            const float s = Q.near2(P.e);
            bool c = P.id >= 0 && s <= thr;
            if (METRIC == OMPL_AMD_METRIC_SE3) c = c && !certainly_above<METRIC, DIM>(P.e, Q.q, r);
            if (__ballot(c) == 0) return;
            const float d = Q.finish(P.e, s);
            c = c && d <= r;
            const u64 m = __ballot(c);
            const int64_t place = found + __popcll(m & (((u64)1 << lane) - 1));
            if (c && place < room) (out ? out : (uint64_t *)mine)[place] = pack_key(d, P.id);
            found += __popcll(m);
        };
        for (int64_t p = t.m; p < t.n; p += kTile) {
            TilePoints<DIM> P;
            P.load_tail(t, p, lane);
            add(P);
        }
        const int64_t tiles = (t.m + kTile - 1) / kTile, nodes = (tiles + kTile - 1) / kTile,
                      supers = (nodes + kTile - 1) / kTile;
        auto within = [&](const float *b, int64_t count) -> u64 {
            return __ballot(lane < count && Q.box2(b, lane) <= thr);
        };
        for (int64_t s0 = 0; s0 < supers; s0 += 64) {
            u64 open2 = supers == 1 ? 1ull : within(t.b2 + (s0 >> 6) * NODE, supers - s0);
            for (; open2; open2 &= open2 - 1) {
                const int64_t sn = s0 + __builtin_ctzll(open2), n0 = sn * kTile;
                u64 open1 = nodes == 1 ? 1ull : within(t.b1 + sn * NODE, nodes - n0);
                for (; open1; open1 &= open1 - 1) {
                    const int64_t node = n0 + __builtin_ctzll(open1), t0 = node * kTile;
                    u64 open0 = within(t.b0 + node * NODE, tiles - t0);
                    if (!open0) continue;
                    TilePoints<DIM> P[2];
                    P[0].load(t, t0 + __builtin_ctzll(open0), lane);
                    for (open0 &= open0 - 1;; open0 &= open0 - 1) {
                        if (open0) P[1].load(t, t0 + __builtin_ctzll(open0), lane);
                        add(P[0]);
                        if (!open0) break;
                        P[0] = P[1];
                    }
                }
            }
        }
    }
    if (A.offsets) return;
    if (lane == 0) A.counts[qi] = found;
    if (A.slot_cap && found > 0) {
        // the lanes wrote the slot for each other
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        u64 key = lane < found ? mine[lane] : ~0ull;
        if (found <= 16) key = wave_sort<16>(key, lane);
        else key = wave_sort<64>(key, lane);
        if (lane < found && lane < A.slot_cap) A.keys[qi * A.slot_cap + lane] = key;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

size_t up256(size_t b)
{
    return (b + 255) / 256 * 256;
}

int64_t ceil_div(int64_t a, int64_t b)
{
    return (a + b - 1) / b;
}

unsigned blocks_of(int64_t n, int64_t per)
{
    return (unsigned)ceil_div(n, per);
}

// Room for a radix sort of n pairs of 32-bit words with alternate buffers: it
// sorts small inputs by merging, through a third copy of the pairs.
size_t sort_bytes(int64_t n)
{
    return up256((size_t)n * 16) + ((size_t)1 << 20);
}

// Working space of a build of up to n points.
size_t build_bytes(int64_t n)
{
    return up256(sizeof(TreePlan)) + up256((size_t)(max_buckets(n) + 1) * 4) + 2 * up256((size_t)n * 8) +
           up256((size_t)n * 4);
}

} // namespace

bool tree_supported(int metric, int dim)
{
    return metric == OMPL_AMD_METRIC_SE3 || dim <= kTreeDimMax;
}

void tree_reserve(NNTree &t, int64_t cap, int dim, int tdim)
{
    tree_free(t);
    const int64_t tiles = ceil_div(cap, kTile), nodes = ceil_div(tiles, kTile), supers = ceil_div(nodes, kTile);
    const size_t box = (size_t)2 * tdim * kTile * sizeof(float);
    const size_t sp = up256((size_t)tiles * dim * kTile * sizeof(float)), sid = up256((size_t)tiles * kTile * 4),
                 pos = up256((size_t)cap * 4), b0 = up256((size_t)nodes * box), b1 = up256((size_t)supers * box),
                 b2 = up256((size_t)ceil_div(supers, kTile) * box);
    t.block = take_block(sp + sid + pos + b0 + b1 + b2 + build_bytes(cap));
    t.mem = (char *)t.block.p;
    char *at = t.mem;
    auto take = [&](size_t b) {
        char *r = at;
        at += b;
        return r;
    };
    t.sp = (float *)take(sp);
    t.sid = (int32_t *)take(sid);
    t.pos = (int32_t *)take(pos);
    t.b0 = (float *)take(b0);
    t.b1 = (float *)take(b1);
    t.b2 = (float *)take(b2);
    t.build = at;
    t.cap = cap;
}

void tree_free(NNTree &t)
{
    give_block(t.block);
    t = NNTree{};
}

void tree_build(NNTree &t, const float *pts, const uint8_t *removed, uint32_t *live, int64_t n, int dim, int tdim,
                hipStream_t s)
{
    OA_REQUIRE(n >= kSample && n <= t.cap, OMPL_AMD_ERR_INTERNAL, "index build out of range");
    const int64_t tiles = ceil_div(n, kTile), nodes = ceil_div(tiles, kTile), supers = ceil_div(nodes, kTile);
    const int64_t buckets = max_buckets(n);
    char *at = t.build;
    auto take = [&](size_t b) {
        char *r = at;
        at += up256(b);
        return r;
    };
    TreePlan *plan = (TreePlan *)take(sizeof(TreePlan));
    uint32_t *counts = (uint32_t *)take((size_t)(buckets + 1) * 4);
    uint2 *place = (uint2 *)take((size_t)n * 8);
    unsigned long long *keys = (unsigned long long *)take((size_t)n * 8);
    uint32_t *perm = (uint32_t *)take((size_t)n * 4);
    const unsigned sweep = (unsigned)std::min<int64_t>(ceil_div(n, 1024), 256);
    if (n < kSmallPoints)
        hipLaunchKernelGGL(tree_sample_kernel<kSmallSample>, dim3((unsigned)tdim), dim3(kSmallSample / 4), 0, s, pts, n,
                           dim, plan);
    else
        hipLaunchKernelGGL(tree_sample_kernel<kSample>, dim3((unsigned)tdim), dim3(kSample / 4), 0, s, pts, n, dim, plan);
    hipLaunchKernelGGL(plan_kernel, dim3(1), dim3(256), 0, s, n, tdim, plan, counts, buckets);
    hipLaunchKernelGGL(tree_buckets_kernel, dim3(sweep), dim3(1024), 0, s, pts, n, dim, tdim, plan, counts, place);
    hipLaunchKernelGGL(tree_scan_kernel, dim3(1), dim3(1024), 0, s, counts, buckets);
    hipLaunchKernelGGL(tree_scatter_kernel, dim3(blocks_of(n, 256)), dim3(256), 0, s, pts, n, dim, tdim, counts,
                       place, keys);
    hipLaunchKernelGGL(tree_sort_kernel, dim3((unsigned)(buckets + ceil_div(n, kBucketSort))), dim3(256), 0, s, plan,
                       tdim, buckets, counts, keys, perm);
    hipLaunchKernelGGL(tree_gather_kernel, dim3(blocks_of(tiles, 4)), dim3(256), 0, s, pts, removed, n, dim, tdim,
                       tiles, perm, t, live);
    hipLaunchKernelGGL(tree_boxes_kernel, dim3(blocks_of(nodes, 4)), dim3(256), 0, s, t.b0, tiles, t.b1, nodes, tdim);
    if (supers > 1) // a single supernode's box is never looked at
        hipLaunchKernelGGL(tree_boxes_kernel, dim3(blocks_of(supers, 4)), dim3(256), 0, s, t.b1, nodes, t.b2, supers,
                           tdim);
    OA_HIP(hipGetLastError());
    t.m = n;
}

void tree_remove(const NNTree &t, int64_t id, hipStream_t s)
{
    if (id >= t.m) return;
    hipLaunchKernelGGL(tree_remove_kernel, dim3(1), dim3(64), 0, s, t.pos, t.sid, id);
    OA_HIP(hipGetLastError());
}

// Radius queries are ordered when there are enough of them to share what they
// read and the points do not fit one XCD's 4 MiB L2 (150,000 of seven coordinates;
// measured at one size: points of fewer would fit up to more): 65,536 queries of 1,000,000
// SE3 points took 430 us in the caller's order and 190 us in this one (reads
// bound it), for 40 us of ordering.  k-NN batches are not: their time is
// instructions, and ordering (40-60 us) gained at most as much (705 us without,
// 711 with, same sizes).
size_t tree_order_bytes(const NNTree &t, int64_t nq)
{
    if (nq < 16384 || t.m < 150000 || nq > INT32_MAX) return 0;
    return 4 * up256((size_t)nq * 4) + sort_bytes(nq);
}

const uint32_t *tree_order(const NNTree &t, const float *q, int64_t nq, int dim, int tdim, void *scratch,
                           hipStream_t s)
{
    char *at = (char *)scratch;
    const size_t each = up256((size_t)nq * 4);
    hipcub::DoubleBuffer<uint32_t> keys((uint32_t *)at, (uint32_t *)(at + each));
    hipcub::DoubleBuffer<uint32_t> perm((uint32_t *)(at + 2 * each), (uint32_t *)(at + 3 * each));
    size_t tmp_bytes = sort_bytes(nq);
    const int bits = std::min(8, 24 / tdim);
    hipLaunchKernelGGL(query_keys_kernel, dim3(blocks_of(nq, 256)), dim3(256), 0, s, (const TreePlan *)t.build,
                       bits, q, nq, dim, tdim, keys.Current(), perm.Current());
    OA_HIP(hipcub::DeviceRadixSort::SortPairs(at + 4 * each, tmp_bytes, keys, perm, (int)nq, 0, bits * tdim, s));
    return perm.Current();
}

// Waves per query: one when the batch alone fills the device, more for smaller
// batches, whose time is their longest query's chain of reads (in 4 and more
// dimensions the queries differ widely: `heavy`).  Measured with 1 / 2 / 4 / 16
// waves, k = 10: 64 queries of 100,000 in R^7 81 / 57 / 40 / 30 us, 1,024:
// 93 / 64 / 48 / 104, 4,096: 105 / 89 / 105 / 343, 16,384: 246 / 269 / 352 /
// 1,329; 4,096 of 100,000 in R^3 25 / 33 / 45 / 200.
static int waves_per_query(int64_t nq, bool heavy)
{
    return nq > 6144 ? 1 : nq > 2048 ? (heavy ? 2 : 1) : nq > 128 ? 4 : 16;
}

template <int METRIC, int DIM, int W>
static void launch_knn_waves(const TreeKnnArgs &A, hipStream_t s)
{
    const dim3 grid(W == 1 ? blocks_of(A.nq, 4) : (unsigned)A.nq), block(W == 1 ? 256 : 64 * W);
    if (A.t.live) hipLaunchKernelGGL((tree_knn_kernel<METRIC, DIM, W, true>), grid, block, 0, s, A);
    else hipLaunchKernelGGL((tree_knn_kernel<METRIC, DIM, W, false>), grid, block, 0, s, A);
}

template <int METRIC, int DIM>
static void launch_knn(const TreeKnnArgs &A, hipStream_t s)
{
    switch (waves_per_query(A.nq, DIM > 3)) {
    case 1:
        launch_knn_waves<METRIC, DIM, 1>(A, s);
        break;
    case 2:
        launch_knn_waves<METRIC, DIM, 2>(A, s);
        break;
    case 4:
        launch_knn_waves<METRIC, DIM, 4>(A, s);
        break;
    default:
        launch_knn_waves<METRIC, DIM, 16>(A, s);
        break;
    }
}

#define OA_TREE_DIMS(X) X(1) X(2) X(3) X(4) X(5) X(6) X(7)

void tree_knn(int metric, int dim, const TreeKnnArgs &A, hipStream_t s)
{
    if (metric == OMPL_AMD_METRIC_SE3) {
        launch_knn<OMPL_AMD_METRIC_SE3, 7>(A, s);
    } else {
#define OA_CASE(D)                                                                                                   \
    if (dim == D) launch_knn<OMPL_AMD_METRIC_L2, D>(A, s);
        OA_TREE_DIMS(OA_CASE)
#undef OA_CASE
    }
    OA_HIP(hipGetLastError());
}

void tree_radius(int metric, int dim, const TreeRadiusArgs &A, hipStream_t s)
{
    const dim3 grid(blocks_of(A.nq, 4)), block(256);
    if (metric == OMPL_AMD_METRIC_SE3) {
        hipLaunchKernelGGL((tree_radius_kernel<OMPL_AMD_METRIC_SE3, 7>), grid, block, 0, s, A);
    } else {
#define OA_CASE(D)                                                                                                   \
    if (dim == D) hipLaunchKernelGGL((tree_radius_kernel<OMPL_AMD_METRIC_L2, D>), grid, block, 0, s, A);
        OA_TREE_DIMS(OA_CASE)
#undef OA_CASE
    }
    OA_HIP(hipGetLastError());
}

} // namespace ompl_amd
