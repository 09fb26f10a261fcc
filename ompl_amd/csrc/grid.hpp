// Cell grid of an environment: for every cell of the arm's workspace, what the
// obstacles can be to a robot sphere centred in it.  Built once with the
// environment (grid.hip); grid_check.hip's kernels read it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "arm_device.hpp"

namespace ompl_amd {

// Cell words.  Top byte 0: no obstacle touches a robot sphere centred in the
// cell, nor one centred up to word / kClearUnits metres from any point of it (the
// cell's clearance).  kCellHit: some obstacle touches every such sphere;
// kCellScan: any obstacle may; else the obstacles that may, their count in the
// top byte: one or two as 12-bit numbers below it (id | id << 12), three to 253
// as the offset of their list.  Only those spheres need an exact test.
constexpr uint32_t kCellHit = 0xffffffffu, kCellScan = 0xfe000000u, kCellNamed = 1u << 24;
constexpr int kCellList = 253; // most obstacles of a list
constexpr float kClearUnits = 4096.0f, kClearMost = 2.0f;
// Distances from a link's second sphere to its fourth, the farthest, and to
// its neighbours; as clearances (units, with 1e-4 m for the rounding of centres)
// from which a second sphere clears the whole link, and all but its last sphere.
constexpr float kFarReach = 0.15f, kClearReach = 0.075f;
constexpr uint32_t kFarUnits = (uint32_t)((kFarReach + 1e-4f) * kClearUnits) + 1,
                   kClearReachUnits = (uint32_t)((kClearReach + 1e-4f) * kClearUnits) + 1;

struct GridView {
    const uint32_t *cells; // [nx][ny][nz]
    const uint16_t *lists; // obstacle numbers
    // obstacle i: tab[2 i] = (lo.xyz, squared contact distance), tab[2 i + 1] =
    // (hi.xyz, 0); a sphere is the box lo = hi = its centre
    const float4 *tab;
    int n_obs;
    int nx, ny, nz;
    float ox, oy, oz, inv; // corner, cells per metre
    float sx, sy, sz;      // -corner * inv: cell coordinate = x inv + sx
    int base_hit;          // an obstacle touches the arm's base link, which never moves
};

// Extents and cell counts for obstacles given as (lo, hi) boxes grown by their
// contact distance; leaves everything else of the view alone.
void grid_extent(GridView &g, const double lo[3], const double hi[3], bool empty);
// Bytes of the cells and the lists of a grid of g's size (cells first, 256-byte aligned).
size_t grid_cells_bytes(const GridView &g);
size_t grid_lists_bytes(const GridView &g);
// Fills cells and lists; counter: one device word of scratch; base: where the
// kernel stores the view's base_hit (device-visible).
void launch_grid_build(const GridView &g, uint32_t *cells, uint16_t *lists, uint32_t *counter, int *base,
                       hipStream_t s);

} // namespace ompl_amd
