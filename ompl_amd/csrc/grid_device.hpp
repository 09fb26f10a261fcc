// State checks over an environment's cell grid (grid.hpp), for one state per
// lane and for eight lanes per state.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "grid.hpp"
#include "walk_device.hpp"

namespace ompl_amd {

__device__ __forceinline__ uint32_t cell_word(const GridView &g, float x, float y, float z)
{
    // outside the grid: the border cell (for NaN: some cell)
    const int ix = (int)__builtin_amdgcn_fmed3f(__builtin_fmaf(x, g.inv, g.sx), 0.0f, (float)(g.nx - 1));
    const int iy = (int)__builtin_amdgcn_fmed3f(__builtin_fmaf(y, g.inv, g.sy), 0.0f, (float)(g.ny - 1));
    const int iz = (int)__builtin_amdgcn_fmed3f(__builtin_fmaf(z, g.inv, g.sz), 0.0f, (float)(g.nz - 1));
    return g.cells[(ix * g.ny + iy) * g.nz + iz];
}

// Exact test of a sphere against one obstacle.
__device__ __forceinline__ bool obstacle_hit(const GridView &g, int o, float x, float y, float z)
{
    const float4 lo = g.tab[2 * o], hi = g.tab[2 * o + 1];
    const float dx = x - clamp_box(x, lo.x, hi.x), dy = y - clamp_box(y, lo.y, hi.y), dz = z - clamp_box(z, lo.z, hi.z);
    return (dx * dx + dy * dy) + dz * dz < lo.w;
}

// Pending exact tests of one wave, in LDS: a state has a few, at different
// spheres in different lanes, so tested where they arise they would cost the
// wave a round trip for each of its 24 spheres; collected, 64 of them share one.
struct WaveTests {
    static constexpr int kRoom = 64 + 4 * 64; // fewer than 64 waiting, and one link's four spheres
    float4 item[kRoom];                       // centre, cell word
    uint8_t owner[kRoom];                     // lane
    uint32_t hit[2];                          // lanes with a hit
};

struct Tests {
    const GridView &g;
    WaveTests &w;
    int n = 0; // wave-uniform
    __device__ __forceinline__ Tests(const GridView &grid, WaveTests &lds) : g(grid), w(lds)
    {
        if (lane_id() < 2) w.hit[lane_id()] = 0;
    }
    __device__ __forceinline__ void sync()
    {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    // Runs the waiting tests, one per lane; true for the lanes that have had a hit.
    __device__ __forceinline__ bool drain()
    {
        const int lane = lane_id();
        sync();
#pragma unroll 1
        for (int i = lane; i < n; i += 64) {
            const float4 t = w.item[i];
            const uint32_t wd = __float_as_uint(t.w), owner = w.owner[i];
            const bool scan = wd == kCellScan;
            const int m = scan ? g.n_obs : (int)(wd >> 24);
#pragma unroll 1
            for (int k = 0; k < m; ++k) { // once, but for a cell in twenty
                // (a scan of one or two obstacles, too, goes by k: its word names none)
                int o = scan ? k : (int)(wd >> (k == 0 ? 0 : 12)) & 0xfff;
                if (!scan && m > 2) o = (int)g.lists[(wd & 0xffffffu) + k];
                if (obstacle_hit(g, o, t.x, t.y, t.z)) {
                    atomicOr(&w.hit[owner >> 5], 1u << (owner & 31));
                    break;
                }
            }
        }
        n = 0;
        sync();
        return (w.hit[lane >> 5] >> (lane & 31)) & 1u;
    }
    // One sphere (at p + Z off) of each `look` lane in a cell with word wd.
    __device__ __forceinline__ void sphere(bool look, uint32_t wd, const float p[3], const float Z[3], float off)
    {
        const bool c = look && wd >= kCellNamed;
        const uint64_t m = wave_ballot(c);
        if (m == 0) return;
        const int lane = lane_id();
        if (c) {
            const int at = n + __popcll(m & (((uint64_t)1 << lane) - 1));
            w.item[at] = make_float4(p[0] + Z[0] * off, p[1] + Z[1] * off, p[2] + Z[2] * off, __uint_as_float(wd));
            w.owner[at] = (uint8_t)lane;
        }
        n += __popcll(m);
    }
};

// The cells speak for centres within the workspace: sincos_pl is a sine and
// cosine below 6000 rad only, so a state beyond (or not a number) is tested
// against every obstacle.
__device__ __forceinline__ bool odd_state(const float q[kDof])
{
    float m = 0.0f;
    bool nan = false;
#pragma unroll
    for (int j = 0; j < kDof; ++j) {
        m = fmaxf(m, fabsf(q[j]));
        nan = nan || q[j] != q[j];
    }
    return nan || !(m < 6000.0f);
}

// Clearance of a cell, in units; 0 where an obstacle may touch a sphere.
__device__ __forceinline__ uint32_t clearance(uint32_t word)
{
    return word < kCellNamed ? word : 0u;
}

__device__ __forceinline__ bool at_least(uint32_t word, uint32_t clear)
{
    return word - clear < kCellNamed - clear;
}

// How fast a motion's spheres move, for turning clearances into positions.
struct Speeds {
    float steps[kDof - 1]; // positions that link 1 .. 6 needs for one unit of clearance
    uint32_t far, near;    // clearances of a second sphere that spare the look at the others
};

// One state per lane.  CLEAR: also how many positions before and after this one
// are certainly valid if it is (`steps`), as far as the cells tell.
template <bool CLEAR = false>
__device__ __forceinline__ bool state_hit1(const GridView &g, const float q[kDof], bool live, WaveTests &lds,
                                           const Speeds &sp = {}, float *steps = nullptr)
{
    if (CLEAR) *steps = 0.0f;
    if (g.base_hit) return live;
    const uint32_t far = CLEAR ? sp.far : kFarUnits, near = CLEAR ? sp.near : kClearReachUnits;
    const bool odd = odd_state(q);
    float X[3] = {1.0f, 0.0f, 0.0f}, Y[3] = {0.0f, 1.0f, 0.0f}, Z[3] = {0.0f, 0.0f, 1.0f}, p[3] = {0.0f, 0.0f, 0.0f};
    float P[kDof - 1][3], W[kDof - 1][3];
    uint32_t w[kDof - 1];
#pragma unroll
    for (int i = 0; i < kDof; ++i) {
        float s, c;
        sincos_pl(q[i], s, c);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if ((i & 1) == 0) {
                const float nx = X[k] * c + Y[k] * s, ny = Y[k] * c - X[k] * s;
                X[k] = nx;
                Y[k] = ny;
            } else {
                const float nx = X[k] * c - Z[k] * s, nz = X[k] * s + Z[k] * c;
                X[k] = nx;
                Z[k] = nz;
            }
        }
        if (i > 0) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                P[i - 1][k] = p[k];
                W[i - 1][k] = Z[k];
            }
            // the reads of all links are in flight together
            w[i - 1] = cell_word(g, p[0] + Z[0] * sphere_offset(1), p[1] + Z[1] * sphere_offset(1),
                                 p[2] + Z[2] * sphere_offset(1));
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) p[k] = p[k] + Z[k] * kLink;
    }
    bool hit = false;
#pragma unroll
    for (int i = 0; i + 1 < kDof; ++i) {
        if (odd) w[i] = kCellScan;
        hit = hit || w[i] == kCellHit;
    }
    if (wave_ballot(live && !hit) == 0) return hit && live;
    // the other spheres of the links that are not far from everything
    uint32_t v[kDof - 1][4];
#pragma unroll
    for (int i = 0; i + 1 < kDof; ++i) {
        const uint32_t c = w[i];
        const bool look = live && !hit && !at_least(c, far);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            // a sphere that is not looked at has at least what is left of the second's
            v[i][m] = m == 1 ? w[i] : c - (m == 3 ? kFarUnits : kClearReachUnits);
            if (m != 1 && look && (m == 3 || !at_least(c, near)))
                v[i][m] = odd ? kCellScan
                              : cell_word(g, P[i][0] + W[i][0] * sphere_offset(m),
                                          P[i][1] + W[i][1] * sphere_offset(m),
                                          P[i][2] + W[i][2] * sphere_offset(m));
        }
    }
#pragma unroll
    for (int i = 0; i + 1 < kDof; ++i) hit = hit || v[i][0] == kCellHit || v[i][2] == kCellHit || v[i][3] == kCellHit;
    if (wave_ballot(live && !hit) == 0) return hit && live;
    if (CLEAR) {
        float least = INFINITY;
#pragma unroll
        for (int i = 0; i + 1 < kDof; ++i) {
            uint32_t c = clearance(v[i][0]);
#pragma unroll
            for (int m = 1; m < 4; ++m) c = min(c, clearance(v[i][m]));
            least = fminf(least, (float)c * sp.steps[i]);
        }
        *steps = odd ? 0.0f : least;
    }
    // the few centres that are tested are made again from the frames: kept, all
    // 24 would take 72 registers
#pragma unroll
    for (int i = 0; i + 1 < kDof; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) asm volatile("" : "+v"(P[i][k]), "+v"(W[i][k]));
    Tests T(g, lds);
#pragma unroll
    for (int i = 0; i + 1 < kDof; ++i) {
        const bool look = live && !hit;
#pragma unroll
        for (int m = 0; m < 4; ++m) T.sphere(look, v[i][m], P[i], W[i], sphere_offset(m));
        if (T.n >= 64 || (i + 2 == kDof && T.n > 0)) hit = T.drain() || hit;
    }
    return hit && live;
}

// Eight lanes per state, lane j of the group holding joint j (qj) and link j:
// the lane's result (the state's is the OR over the group).
__device__ __forceinline__ bool state_hit8(const GridView &g, float qj, bool live, WaveTests &lds)
{
    if (g.base_hit) return live;
    const int j = threadIdx.x & 7, group = threadIdx.x & 56;
    const bool odd = ((wave_ballot(j < kDof && !(fabsf(qj) < 6000.0f)) >> group) & 0x7f) != 0;
    float sm, cm, p[3], Z[3];
    sincos_pl(qj, sm, cm);
    link_chain<8>(sm, cm, j, p, Z);
    const bool mine = live && j > 0 && j < kDof;
    uint32_t w[4];
    // the link's cells are read together: one round trip
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        w[m] = 0;
        if (mine)
            w[m] = odd ? kCellScan
                       : cell_word(g, p[0] + Z[0] * sphere_offset(m), p[1] + Z[1] * sphere_offset(m),
                                   p[2] + Z[2] * sphere_offset(m));
    }
    bool hit = w[0] == kCellHit || w[1] == kCellHit || w[2] == kCellHit || w[3] == kCellHit;
    const bool done = ((wave_ballot(hit) >> group) & 0xff) != 0;
    if (wave_ballot(mine && !done) == 0) return hit;
    Tests T(g, lds);
#pragma unroll
    for (int m = 0; m < 4; ++m) T.sphere(mine && !done, w[m], p, Z, sphere_offset(m));
    if (T.n) hit = T.drain() || hit;
    return hit;
}

} // namespace ompl_amd
