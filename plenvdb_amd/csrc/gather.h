// Trilinear sampling helpers shared by the per-point kernels and the fused
// step: the reference's corner walk, the cell decomposition and a one-entry
// leaf cache (the analogue of the ReadAccessor's leaf-level cache).
#pragma once

#include "pvdb_common.h"

namespace pvdb {

// Corner walk of the reference: 000,001,011,010,110,111,101,100
// (plenvdb/lib/vdb/densityvdb.cu:115-122).  Bit q of each mask is the corner's
// x/y/z offset.
constexpr unsigned kCx = 0xF0u, kCy = 0x3Cu, kCz = 0x66u;

struct Cell {
    int i0, j0, k0;
    float u, v, w;
};

__device__ __forceinline__ Cell make_cell(float x, float y, float z) {
    Cell c;
    c.i0 = (int)floorf(x);
    c.j0 = (int)floorf(y);
    c.k0 = (int)floorf(z);
    c.u = x - (float)c.i0;
    c.v = y - (float)c.j0;
    c.w = z - (float)c.k0;
    return c;
}

// One-entry leaf cache, the analogue of the accessor's leaf-level cache.
struct LeafCache {
    int key0, key1, key2;
    int32_t leaf;
    __device__ __forceinline__ LeafCache() : key0(INT32_MIN), key1(0), key2(0), leaf(-1) {}
    __device__ __forceinline__ int64_t slot(const TopoView& t, int i, int j, int k) {
        const int a = i >> 3, b = j >> 3, c = k >> 3;
        if (a != key0 || b != key1 || c != key2) {
            key0 = a;
            key1 = b;
            key2 = c;
            leaf = pvdb::leaf_of(t, i, j, k);
        }
        return leaf < 0 ? int64_t(-1) : (int64_t)leaf * 512 + pvdb::voxel_offset(i, j, k);
    }
};


// leaf_of with a selected index instead of a branch around the load, for a table
// that exists (uniform: the one-level layout of a topology with leaves).
__device__ __forceinline__ bool one_level(const TopoView& t) { return !t.two_level && t.nleaf > 0; }
__device__ __forceinline__ int32_t leaf_at(const TopoView& t, int i, int j, int k) {
    const int a = (i >> 3) - t.lo0, b = (j >> 3) - t.lo1, c = (k >> 3) - t.lo2;
    const bool in = (unsigned)a < (unsigned)t.d0 && (unsigned)b < (unsigned)t.d1 &&
                    (unsigned)c < (unsigned)t.d2;
    const int32_t l = t.table[in ? ((int64_t)a * t.d1 + b) * t.d2 + c : 0];
    return in ? l : -1;
}

// Whether a corner of the cell can lie in the leaf table's box.
__device__ __forceinline__ bool near_leaves(const TopoView& t, const Cell& cell) {
    return (unsigned)((cell.i0 >> 3) - t.lo0 + 1) <= (unsigned)t.d0 &&
           (unsigned)((cell.j0 >> 3) - t.lo1 + 1) <= (unsigned)t.d1 &&
           (unsigned)((cell.k0 >> 3) - t.lo2 + 1) <= (unsigned)t.d2;
}

// Slots (-1: no leaf) of the cell's corners, in corner order.  The eight lookups do
// not depend on one another, so a sample waits for the leaf table once, and for its
// values once: with a leaf cache walked corner by corner each value was waited for
// before the next corner's lookup.  The forward march of 8192 rays 19.6 -> 15.2 us, of 1021
// 13.5 -> 10.2; k_direct_composite (3 channels, 8192 rays) 21.4 -> 17.0; the point
// gather of 1.2M densities 14.6 -> 11.3, of 200k 12-channel rows 12.0 -> 9.3.
//
// kAnywhere: the points of a query, which may lie far from any leaf and are many at a
// time, look up one leaf unless their cell crosses into others, and none outside the
// table's box.  4M densities all over a grid of 600 leaves 37.7 us (leaf cache), 56.4
// (eight lookups a point), 34.4; none of them near a leaf 21.1, 27.6, 17.1; along rays
// 36.4, 30.0, 30.6.  A march's samples lie in leaves, and wait less without the branches
// (8192 rays, coarse stage: 69.6 us a step, 71.8 with them).
template <bool kAnywhere>
__device__ __forceinline__ void corner_slots(const TopoView& t, const Cell& cell, int64_t (&s)[8]) {
    if (one_level(t)) {  // uniform
        int32_t l[8];
        if constexpr (kAnywhere) {
#pragma unroll
            for (int q = 0; q < 8; ++q) l[q] = -1;
            if (near_leaves(t, cell)) {
                const int32_t l0 = leaf_at(t, cell.i0, cell.j0, cell.k0);
                const bool cross =
                    (cell.i0 & 7) == 7 || (cell.j0 & 7) == 7 || (cell.k0 & 7) == 7;
                if (cross) {  // the other seven, without a wait for the first
#pragma unroll
                    for (int q = 1; q < 8; ++q)
                        l[q] = leaf_at(t, cell.i0 + ((kCx >> q) & 1), cell.j0 + ((kCy >> q) & 1),
                                       cell.k0 + ((kCz >> q) & 1));
                }
                l[0] = l0;
#pragma unroll
                for (int q = 1; q < 8; ++q) l[q] = cross ? l[q] : l0;
            }
        } else {
#pragma unroll
            for (int q = 0; q < 8; ++q)
                l[q] = leaf_at(t, cell.i0 + ((kCx >> q) & 1), cell.j0 + ((kCy >> q) & 1),
                               cell.k0 + ((kCz >> q) & 1));
        }
#pragma unroll
        for (int q = 0; q < 8; ++q)
            s[q] = l[q] < 0 ? int64_t(-1)
                            : (int64_t)l[q] * 512 + voxel_offset(cell.i0 + ((kCx >> q) & 1),
                                                                 cell.j0 + ((kCy >> q) & 1),
                                                                 cell.k0 + ((kCz >> q) & 1));
        return;
    }
    LeafCache cache;
#pragma unroll
    for (int q = 0; q < 8; ++q)
        s[q] = cache.slot(t, cell.i0 + ((kCx >> q) & 1), cell.j0 + ((kCy >> q) & 1),
                          cell.k0 + ((kCz >> q) & 1));
}

// The cell's fractions towards corner q.
__device__ __forceinline__ void corner_fracs(const Cell& cell, int q, float& a, float& b, float& d) {
    a = ((kCx >> q) & 1) ? cell.u : 1.f - cell.u;
    b = ((kCy >> q) & 1) ? cell.v : 1.f - cell.v;
    d = ((kCz >> q) & 1) ? cell.w : 1.f - cell.w;
}

// Whether a point's corner values are loaded: a point of a query's, when it has any;
// else when there are leaves at all (uniform).  Without, its corners weigh zeros, so that
// a coordinate that is not finite gives NaN as with them.
template <bool kAnywhere>
__device__ __forceinline__ bool has_values(const TopoView& t, const int64_t (&s)[8]) {
    if constexpr (!kAnywhere) return t.nleaf > 0;
    bool any = false;
#pragma unroll
    for (int q = 0; q < 8; ++q) any = any || s[q] >= 0;
    return any;
}

// Density at an index-space point, density rule of densityvdb.cu:115-122.  With NO
// slot, slot 0's value is loaded in its place.
template <bool kAnywhere = false>
__device__ __forceinline__ float gather_density(const TopoView& t, const float* __restrict__ vals,
                                                const Cell& cell) {
    int64_t s[8];
    corner_slots<kAnywhere>(t, cell, s);
    float v[8], acc = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = 0.f;
    if (has_values<kAnywhere>(t, s)) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = vals[s[q] >= 0 ? s[q] : 0];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        float a, b, d;
        corner_fracs(cell, q, a, b, d);
        acc = acc + (((s[q] >= 0 ? v[q] : 0.f) * a) * b) * d;
    }
    return acc;
}

// NC colour channels at an index-space point, colour rule of
// colorvdb.cu:16-26,96-103: the corner weight (a*b)*c first, then
// out[c] += val[c] * weight, corners in the order above (a missing leaf adds 0).
// kWide: rows are 16-byte aligned (NC a multiple of 4).  At most four corners' rows of
// twelve channels are in registers at a time.
template <int NC, bool kWide = NC % 4 == 0, bool kAnywhere = false>
__device__ __forceinline__ void gather_color(const TopoView& t, const float* __restrict__ vals,
                                             const Cell& cell, float (&out)[NC]) {
    constexpr int kAtOnce = NC > 4 ? 4 : 8;
    int64_t s[8];
    corner_slots<kAnywhere>(t, cell, s);
#pragma unroll
    for (int c = 0; c < NC; ++c) out[c] = 0.f;
    const bool some = has_values<kAnywhere>(t, s);
#pragma unroll
    for (int q0 = 0; q0 < 8; q0 += kAtOnce) {
        float v[kAtOnce][NC];
#pragma unroll
        for (int k = 0; k < kAtOnce; ++k) {
            const float* src = vals + (s[q0 + k] >= 0 ? s[q0 + k] : 0) * NC;
            if (!some) continue;
            if constexpr (kWide) {
#pragma unroll
                for (int e = 0; e < NC / 4; ++e) {
                    const float4 r = reinterpret_cast<const float4*>(src)[e];
                    v[k][4 * e] = r.x;
                    v[k][4 * e + 1] = r.y;
                    v[k][4 * e + 2] = r.z;
                    v[k][4 * e + 3] = r.w;
                }
            } else {
#pragma unroll
                for (int c = 0; c < NC; ++c) v[k][c] = src[c];
            }
        }
#pragma unroll
        for (int k = 0; k < kAtOnce; ++k) {
            float a, b, d;
            corner_fracs(cell, q0 + k, a, b, d);
            const float sc = (a * b) * d;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                out[c] = out[c] + (some && s[q0 + k] >= 0 ? v[k][c] : 0.f) * sc;
        }
    }
}

}  // namespace pvdb
