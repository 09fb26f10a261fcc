// Building an environment's cell grid (grid.hpp).
//
// A cell's word is decided from the least and the greatest distance that a
// point of the cell (grown by kCellMargin) can have from each obstacle.  The
// decisions keep a margin of 1e-4 m and 1e-5 of the contact distance from the
// exact test's threshold, far above the FP32 rounding of centres and distances
// of a 2.1 m arm (a few 1e-7 m), so a cell that says free or hit never
// disagrees with the exact test of a sphere centred in it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "grid.hpp"
#include "walk_device.hpp"

namespace ompl_amd {

namespace {
// Cells along the longest side.  Finer cells leave fewer exact tests but a
// larger table: 64^3 words are 1 MiB, which stays in an XCD's 4 MiB L2.
constexpr int kGridCells = 64;
// Half side of the workspace: no robot sphere's centre is farther than 2.0625
// from the base in any coordinate.
constexpr double kReach = 2.12;
// A cell is grown by this much before it is decided: far more than the rounding
// of a coordinate's cell number (a few 1e-7 of 68 cells of 0.06 m at most).
constexpr float kCellMargin = 1e-4f;
// Margins of the decisions, in metres and of the contact distance.
constexpr float kBoundAbs = 1e-4f, kBoundRel = 1e-5f;

size_t up256(size_t b)
{
    return (b + 255) / 256 * 256;
}

size_t list_entries(const GridView &g)
{
    return std::max<size_t>((size_t)g.nx * g.ny * g.nz * 2, 65536);
}
} // namespace

void grid_extent(GridView &g, const double lo[3], const double hi[3], bool empty)
{
    double a[3], b[3], longest = 0.0;
    bool none = empty;
    for (int k = 0; k < 3; ++k) {
        a[k] = std::max(lo[k], -kReach);
        b[k] = std::min(hi[k], kReach);
        if (!(a[k] < b[k])) none = true;
        longest = std::max(longest, b[k] - a[k]);
    }
    if (none) { // nothing within reach: one cell, which the build finds far from everything
        // (the obstacles stay: a state beyond the sine's range is tested against them)
        g.nx = g.ny = g.nz = 1;
        g.ox = g.oy = g.oz = 0.0f;
        g.inv = 0.0f;
        g.sx = g.sy = g.sz = 0.0f;
        return;
    }
    // two cells more on each side: a point outside the grid takes the border
    // cell's word, which must then be free (where the workspace ends instead,
    // no point is outside)
    const double h = longest / (kGridCells - 4);
    int n[3];
    for (int k = 0; k < 3; ++k) {
        a[k] -= 2 * h;
        n[k] = std::min(kGridCells + 4, (int)std::ceil((b[k] + 2 * h - a[k]) / h));
    }
    g.nx = n[0];
    g.ny = n[1];
    g.nz = n[2];
    g.ox = (float)a[0];
    g.oy = (float)a[1];
    g.oz = (float)a[2];
    g.inv = (float)(1.0 / h);
    g.sx = (float)(-a[0] / h);
    g.sy = (float)(-a[1] / h);
    g.sz = (float)(-a[2] / h);
}

size_t grid_cells_bytes(const GridView &g)
{
    return up256((size_t)g.nx * g.ny * g.nz * sizeof(uint32_t));
}

size_t grid_lists_bytes(const GridView &g)
{
    return up256(list_entries(g) * sizeof(uint16_t));
}

// Least and greatest distance of obstacle (lo, hi) from the points of the box [a, b].
__device__ __forceinline__ void box_range(const float a[3], const float b[3], float4 lo, float4 hi, float &least,
                                          float &most)
{
    const float l[3] = {lo.x, lo.y, lo.z}, h[3] = {hi.x, hi.y, hi.z};
    float s = 0.0f, t = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float g = fmaxf(fmaxf(l[k] - b[k], a[k] - h[k]), 0.0f);
        const float m = fmaxf(fmaxf(l[k] - a[k], b[k] - h[k]), 0.0f);
        s += g * g;
        t += m * m;
    }
    least = sqrtf(s);
    most = sqrtf(t);
}

// One wave per brick of 4 x 4 x 4 cells, four bricks a block: the wave's lanes
// first pick, 64 at a time, the obstacles that come near the brick, then each
// lane decides its cell against those.
constexpr int kPicked = 512; // obstacles kept per brick; more: its cells are scanned

__global__ void __launch_bounds__(256) grid_build_kernel(GridView g, uint32_t *__restrict__ cells,
                                                         uint16_t *__restrict__ lists, uint32_t entries,
                                                         uint32_t *__restrict__ cursor)
{
    __shared__ uint16_t picked[4][kPicked];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int bx = (g.nx + 3) / 4, by = (g.ny + 3) / 4, bz = (g.nz + 3) / 4;
    const int brick = blockIdx.x * 4 + w;
    if (brick >= bx * by * bz) return; // wave-uniform; the block has no barrier
    const int x0 = brick / (by * bz) * 4, y0 = brick / bz % by * 4, z0 = brick % bz * 4;
    const float h = g.inv > 0.0f ? 1.0f / g.inv : 0.0f;
    auto span = [&](int i, int n, float o, float &a, float &b) {
        a = o + (float)i * h - kCellMargin;
        b = o + (float)(i + n) * h + kCellMargin;
    };
    float a[3], b[3];
    span(x0, 4, g.ox, a[0], b[0]);
    span(y0, 4, g.oy, a[1], b[1]);
    span(z0, 4, g.oz, a[2], b[2]);
    int n = 0;
    bool many = false;
    float rest = kClearMost; // clearance of the brick from the obstacles not picked
    for (int o0 = 0; o0 < g.n_obs; o0 += 64) {
        const int o = o0 + lane;
        bool near = false;
        if (o < g.n_obs) {
            const float4 lo = g.tab[2 * o], hi = g.tab[2 * o + 1];
            float least, most;
            box_range(a, b, lo, hi, least, most);
            const float gap = least - (sqrtf(lo.w) * (1.0f + kBoundRel) + kBoundAbs);
            near = !(gap > kFarReach + kBoundAbs);
            if (!near) rest = fminf(rest, gap);
        }
        const uint64_t m = __ballot(near);
        const int at = n + __popcll(m & (((uint64_t)1 << lane) - 1));
        if (near && at < kPicked) picked[w][at] = (uint16_t)o;
        n += __popcll(m);
    }
    if (n > kPicked) {
        many = true;
        n = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int x = x0 + (lane >> 4), y = y0 + ((lane >> 2) & 3), z = z0 + (lane & 3);
    const bool in = x < g.nx && y < g.ny && z < g.nz;
    span(x, 1, g.ox, a[0], b[0]);
    span(y, 1, g.oy, a[1], b[1]);
    span(z, 1, g.oz, a[2], b[2]);
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) rest = fminf(rest, __shfl_xor(rest, d));
    bool hit = false;
    float clear = rest;
    int count = 0;
    for (int i = 0; i < n; ++i) {
        const int o = picked[w][i];
        const float4 lo = g.tab[2 * o], hi = g.tab[2 * o + 1];
        float least, most;
        box_range(a, b, lo, hi, least, most);
        const float r = sqrtf(lo.w), up = r * (1.0f + kBoundRel) + kBoundAbs, down = r * (1.0f - kBoundRel) - kBoundAbs;
        hit = hit || most < down;
        count += least <= up ? 1 : 0;
        clear = fminf(clear, least - up);
    }
    // (no obstacle within `up`: the least gap is positive)
    uint32_t word = (uint32_t)(fmaxf(clear, 0.0f) * kClearUnits);
    if (hit) word = kCellHit;
    else if (many || count > kCellList) word = kCellScan;
    const bool named = in && !hit && !many && count > 0 && count <= kCellList;
    const int want = named && count > 2 ? count : 0;
    // room for the wave's lists
    int incl = want;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d);
        if (lane >= d) incl += u;
    }
    const int total = __shfl(incl, 63);
    uint32_t base = 0;
    if (total > 0) {
        if (lane == 0) base = atomicAdd(cursor, (uint32_t)total);
        base = (uint32_t)__shfl((int)base, 0);
    }
    if (named) {
        uint32_t at = base + (uint32_t)(incl - want), ids = 0;
        const bool room = (uint64_t)at + (uint64_t)want <= entries && at < (1u << 24) - 512u;
        int k = 0;
        for (int i = 0; i < n; ++i) {
            const int o = picked[w][i];
            const float4 lo = g.tab[2 * o], hi = g.tab[2 * o + 1];
            float least, most;
            box_range(a, b, lo, hi, least, most);
            if (!(least <= sqrtf(lo.w) * (1.0f + kBoundRel) + kBoundAbs)) continue;
            if (want == 0) ids |= (uint32_t)o << (12 * k);
            else if (room) lists[at + k] = (uint16_t)o;
            ++k;
        }
        word = want == 0 || room ? (want == 0 ? ids : at) | (uint32_t)count << 24 : kCellScan;
    }
    if (in) cells[((int64_t)x * g.ny + y) * g.nz + z] = word;
}

// Exact test of the base link's four spheres (one wave).
__global__ void __launch_bounds__(64) grid_base_kernel(GridView g, int *__restrict__ base)
{
    bool hit = false;
    for (int o = threadIdx.x; o < g.n_obs; o += 64) {
        const float4 lo = g.tab[2 * o], hi = g.tab[2 * o + 1];
        for (int m = 0; m < 4; ++m) {
            const float c = 0.0f + 1.0f * sphere_offset(m);
            const float dx = 0.0f - clamp_box(0.0f, lo.x, hi.x), dy = 0.0f - clamp_box(0.0f, lo.y, hi.y),
                        dz = c - clamp_box(c, lo.z, hi.z);
            hit = hit || (dx * dx + dy * dy) + dz * dz < lo.w;
        }
    }
    const uint64_t m = __ballot(hit);
    if (threadIdx.x == 0) *base = m != 0 ? 1 : 0;
}

__global__ void grid_cursor_kernel(uint32_t *cursor)
{
    *cursor = 0;
}

void launch_grid_build(const GridView &g, uint32_t *cells, uint16_t *lists, uint32_t *counter, int *base,
                       hipStream_t s)
{
    const int bricks = ((g.nx + 3) / 4) * ((g.ny + 3) / 4) * ((g.nz + 3) / 4);
    hipLaunchKernelGGL(grid_cursor_kernel, dim3(1), dim3(1), 0, s, counter);
    hipLaunchKernelGGL(grid_build_kernel, dim3((unsigned)((bricks + 3) / 4)), dim3(256), 0, s, g, cells, lists,
                       (uint32_t)list_entries(g), counter);
    hipLaunchKernelGGL(grid_base_kernel, dim3(1), dim3(64), 0, s, g, base);
    OA_HIP(hipGetLastError());
}

} // namespace ompl_amd
