// Spatial index of the nearest-neighbour structure: points in tiles of 64
// that are compact in space, under three levels of bounding boxes with 64
// children each, searched by one wave per query (nn_tree.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "runtime.hpp"

namespace ompl_amd {

constexpr int kTile = 64;   // points per tile, tiles per node, nodes per supernode
// L2 dimensions with an index: up to the arm's.  Boxes exclude less in more: 100,000
// even points, k = 10, 64 / 4,096 / 32,768 queries, full scan against index: 8
// dimensions 149 / 270 / 1,419 against 37 / 149 / 388 us, 10: 148 / 282 / 1,575
// against 47 / 321 / 1,043, 12: 150 / 305 / 1,757 against 81 / 521 / 2,393.
constexpr int kTreeDimMax = 7;
// Points from which on the index is kept.
constexpr int64_t kTreeMinPoints = 2048;

// Device arrays of the index; all in one allocation, sized for `cap` points.
struct NNTree {
    int64_t m = 0;   // points in the index: ids [0, m); later ids are its tail
    int64_t cap = 0; // points the arrays have room for
    DeviceBlock block;
    char *mem = nullptr; // block's
    float *sp = nullptr;       // [tiles][dim][64] coordinates
    int32_t *sid = nullptr;    // [tiles][64] ids; -1: no point, or a removed one
    int32_t *pos = nullptr;    // [cap] place of an id in sid
    float *b0 = nullptr;       // [nodes][2 tdim][64] boxes of a node's tiles (lows, then highs)
    float *b1 = nullptr;       // [supernodes][2 tdim][64] boxes of a supernode's nodes
    float *b2 = nullptr;       // [ceil(supernodes / 64)][2 tdim][64] boxes of the supernodes
    char *build = nullptr;     // the build's own working space (its plan first, kept)
};

// FP32 bits reordered so that unsigned order is numeric order.
__device__ __forceinline__ uint32_t ordered_bits(float v)
{
    const uint32_t u = __float_as_uint(v);
    return u & 0x80000000u ? ~u : u | 0x80000000u;
}

struct TreeView {
    const float *sp;
    const int32_t *sid;
    const float *b0, *b1, *b2;
    int64_t m, n;           // points in the index; all points (ids searched are below n)
    const uint32_t *live;   // a captured k-NN search: where the kernel reads m, since a
                            // replay may find the index built again with more points
    const float *pts;       // [n][dim], the tail is [m, n)
    const uint8_t *removed; // [n]
};

struct TreeKnnArgs {
    TreeView t;
    const float *q; // [nq][dim]
    int64_t nq;
    int k;             // largest k
    const int32_t *kq; // per-query k (clamped to [0, k]), or null
    const int64_t *out_off; // with kq: results of query i at out_off[i]; else at i * k
    float *out_d;
    int32_t *out_i;
};

struct TreeRadiusArgs {
    TreeView t;
    const float *q;
    const uint32_t *order; // the queries in the order they are searched, or null
    int64_t nq;
    float radius;
    const float *rq;  // per-query radius, or null
    int64_t *counts;  // [nq] results per query (written unless `offsets` is given)
    const int64_t *offsets; // write query i's keys from offsets[i] on; null: its first slot_cap keys from i * slot_cap on
    int slot_cap;     // at most 64; 0: count only
    uint64_t *keys;   // distance bits << 32 | id; a slot that holds all of its query's is ascending
};

// Whether (metric, dim) has the index.
bool tree_supported(int metric, int dim);
// Allocates the arrays for `cap` points (the old ones are dropped: m = 0).
void tree_reserve(NNTree &t, int64_t cap, int dim, int tdim);
void tree_free(NNTree &t); // nothing on the device uses the arrays any more
// Indexes points [0, n) of pts ([n][dim]), n >= kTreeMinPoints; removed ones get no entry.
// live: receives n (device).
void tree_build(NNTree &t, const float *pts, const uint8_t *removed, uint32_t *live, int64_t n, int dim, int tdim,
                hipStream_t s);
// Drops id from the index.
void tree_remove(const NNTree &t, int64_t id, hipStream_t s);
// Scratch bytes for tree_order, 0 when the queries are better left in the caller's order.
size_t tree_order_bytes(const NNTree &t, int64_t nq);
// Puts the queries in an order that keeps neighbours together (in scratch).
const uint32_t *tree_order(const NNTree &t, const float *q, int64_t nq, int dim, int tdim, void *scratch,
                           hipStream_t s);
void tree_knn(int metric, int dim, const TreeKnnArgs &A, hipStream_t s);
void tree_radius(int metric, int dim, const TreeRadiusArgs &A, hipStream_t s);

} // namespace ompl_amd
