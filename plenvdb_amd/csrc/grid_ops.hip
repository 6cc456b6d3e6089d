// Per-point and per-slot grid kernels: trilinear gather (forward) and atomic
// scatter (backward) of a VDB payload, dense <-> VDB copies, the VDB Adam step
// and the dense Adam step of the MLP parameters.
//
// These are the kernels behind the reference-compatible plenvdb API (one
// launch per call, reference operation order).  The fused training step lives
// in fused_step.hip.
#include <type_traits>

#include "pvdb_common.h"
#include "gather.h"
#include "plenvdb_hip.h"

namespace pvdb {
TopoView view_of(const pvdb_topology* t);
}

using pvdb::TopoView;
using pvdb::Cell;
using pvdb::LeafCache;
using pvdb::kCx;
using pvdb::kCy;
using pvdb::kCz;
using pvdb::make_cell;

namespace {

// ORDER 0: out += ((val*a)*b)*c          (densityvdb.cu:115-122)
// ORDER 1: out[c] += val[c]*((a*b)*c)    (colorvdb.cu:16-26,96-103)
template <int C, int ORDER>
__global__ void __launch_bounds__(256) k_tri_fwd(TopoView t, const float* __restrict__ vals,
                                                 int cdyn, const float* __restrict__ xs,
                                                 const float* __restrict__ ys,
                                                 const float* __restrict__ zs, int64_t n,
                                                 float* __restrict__ out, int wide) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int CC = C > 0 ? C : cdyn;
    const Cell cell = make_cell(xs[p], ys[p], zs[p]);
    if constexpr (ORDER == 0) {
        out[p] = pvdb::gather_density<true>(t, vals, cell);
        return;
    } else if constexpr (C > 0) {
        float o[C];
        if (C % 4 == 0 && wide)  // uniform
            pvdb::gather_color<C, C % 4 == 0, true>(t, vals, cell, o);
        else
            pvdb::gather_color<C, false, true>(t, vals, cell, o);
#pragma unroll
        for (int c = 0; c < C; ++c) out[p * C + c] = o[c];
        return;
    }
    LeafCache cache;
    float acc[C > 0 ? C : 48];
#pragma unroll
    for (int c = 0; c < (C > 0 ? C : 48); ++c) acc[c] = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int dx = (kCx >> q) & 1, dy = (kCy >> q) & 1, dz = (kCz >> q) & 1;
        const float a = dx ? cell.u : 1.f - cell.u;
        const float b = dy ? cell.v : 1.f - cell.v;
        const float d = dz ? cell.w : 1.f - cell.w;
        const int64_t s = cache.slot(t, cell.i0 + dx, cell.j0 + dy, cell.k0 + dz);
        if (ORDER == 0) {
            const float val = s >= 0 ? vals[s * CC] : 0.f;
            acc[0] = acc[0] + ((val * a) * b) * d;
        } else {
            const float sc = (a * b) * d;
            const float* src = vals + (s >= 0 ? s : 0) * CC;
#pragma unroll
            for (int c = 0; c < (C > 0 ? C : 48); ++c) {
                if (c < CC) {
                    const float val = s >= 0 ? src[c] : 0.f;
                    acc[c] = acc[c] + val * sc;
                }
            }
        }
    }
    float* o = out + p * CC;
#pragma unroll
    for (int c = 0; c < (C > 0 ? C : 48); ++c)
        if (c < CC) o[c] = acc[c];
}

// Scatter with the "leaf must exist" rule (densityvdb.cu:16-27,143-181;
// colorvdb.cu:28-37,130-175): corners in a missing leaf are dropped, voxels of
// existing leaves receive the add whether active or not.
template <int C, int ORDER>
__global__ void __launch_bounds__(256) k_tri_bwd(TopoView t, float* __restrict__ grad, int cdyn,
                                                 const float* __restrict__ xs,
                                                 const float* __restrict__ ys,
                                                 const float* __restrict__ zs,
                                                 const float* __restrict__ g, int64_t n) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int CC = C > 0 ? C : cdyn;
    const Cell cell = make_cell(xs[p], ys[p], zs[p]);
    const float* gp = g + p * CC;
    float gv[C > 0 ? C : 48];
#pragma unroll
    for (int c = 0; c < (C > 0 ? C : 48); ++c) gv[c] = c < CC ? gp[c] : 0.f;
    LeafCache cache;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int dx = (kCx >> q) & 1, dy = (kCy >> q) & 1, dz = (kCz >> q) & 1;
        const float a = dx ? cell.u : 1.f - cell.u;
        const float b = dy ? cell.v : 1.f - cell.v;
        const float d = dz ? cell.w : 1.f - cell.w;
        const int64_t s = cache.slot(t, cell.i0 + dx, cell.j0 + dy, cell.k0 + dz);
        if (s < 0) continue;
        float* dst = grad + s * CC;
        if (ORDER == 0) {
            atomicAdd(dst, ((gv[0] * a) * b) * d);
        } else {
            const float sc = (a * b) * d;
#pragma unroll
            for (int c = 0; c < (C > 0 ? C : 48); ++c)
                if (c < CC) atomicAdd(dst + c, gv[c] * sc);
        }
    }
}

// The same sums as k_tri_bwd with fewer and wider atomics: a workgroup takes 64
// consecutive points (samples of a ray lie half a voxel apart and share most of
// their corners), links the (point, corner) pairs of each slot into a list
// through an LDS hash, and adds every distinct slot's C sums once, a lane per
// channel, so that one request carries a slot's row.  A pair keeps its weight
// only; the walk multiplies it with the point's gradients, which wait in LDS.
// k_tri_bwd is bound by its requests: one per (point, corner, channel), as a
// lane's channels lie in instructions of their own.  200k points along random
// rays, 12 channels: 98.4 -> 15.2 us; 1.2M points, one channel: 33.7 -> 26.2 us;
// 100k samples of rays that all cross one region: 528 -> 27.5 us and, one
// channel, 47.3 -> 12.6 us.  Points in no order, which share no corners, still
// gain by the wide requests.
constexpr int kBwdPoints = 64, kBwdPairs = 8 * kBwdPoints, kBwdSlots = 2 * kBwdPairs;
constexpr uint32_t kNoKey = 0xffffffffu, kNoPair = 0xffffu;

template <int C, int ORDER>
__global__ void __launch_bounds__(256) k_tri_bwd_agg(TopoView t, float* __restrict__ grad,
                                                     const float* __restrict__ xs,
                                                     const float* __restrict__ ys,
                                                     const float* __restrict__ zs,
                                                     const float* __restrict__ g, int64_t n) {
    constexpr int kLanes = C == 12 ? 16 : C == 3 ? 4 : 1;  // lanes per slot in the walk
    __shared__ uint32_t key[kBwdSlots];   // the slot of an entry
    __shared__ uint32_t head[kBwdSlots];  // the entry's first pair
    __shared__ float wgt[kBwdPairs];      // a pair's weight (ORDER 0: its contribution)
    __shared__ uint16_t next[kBwdPairs], listed[kBwdPairs];
    __shared__ float gs[C > 1 ? kBwdPoints * C : 1];
    __shared__ int nlisted;
    const int tid = threadIdx.x;
    const int64_t p0 = (int64_t)blockIdx.x * kBwdPoints;
    const int np = (int)(n - p0 < kBwdPoints ? n - p0 : kBwdPoints);
#pragma unroll
    for (int e = 0; e < kBwdSlots / 256; ++e) {
        key[tid + 256 * e] = kNoKey;
        head[tid + 256 * e] = kNoPair;
    }
    if (tid == 0) nlisted = 0;
    if constexpr (C > 1)
        for (int e = tid; e < np * C; e += 256) gs[e] = g[p0 * C + e];
    int64_t s[2];
    float w[2];
#pragma unroll
    for (int it = 0; it < 2; ++it) {  // pairs tid and tid + 256
        const int pt = (tid >> 3) + 32 * it, q = tid & 7;
        s[it] = -1;
        w[it] = 0.f;
        if (pt < np) {
            const int64_t p = p0 + pt;
            const Cell cell = make_cell(xs[p], ys[p], zs[p]);
            const int dx = (kCx >> q) & 1, dy = (kCy >> q) & 1, dz = (kCz >> q) & 1;
            const float a = dx ? cell.u : 1.f - cell.u;
            const float b = dy ? cell.v : 1.f - cell.v;
            const float d = dz ? cell.w : 1.f - cell.w;
            w[it] = ORDER == 0 ? ((g[p] * a) * b) * d : (a * b) * d;
            s[it] = pvdb::slot_of(t, cell.i0 + dx, cell.j0 + dy, cell.k0 + dz);
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        if (s[it] < 0) continue;
        const int pair = tid + 256 * it;
        wgt[pair] = w[it];
        const uint32_t k = (uint32_t)s[it];
        uint32_t h = (k * 2654435761u) >> 22;  // kBwdSlots == 1 << 10
        while (true) {  // at most kBwdPairs entries: a free one is met
            const uint32_t prev = atomicCAS(&key[h], kNoKey, k);
            if (prev == kNoKey) listed[atomicAdd(&nlisted, 1)] = (uint16_t)h;
            if (prev == kNoKey || prev == k) break;
            h = (h + 1) & (kBwdSlots - 1);
        }
        next[pair] = (uint16_t)atomicExch(&head[h], (uint32_t)pair);
    }
    static_assert(kBwdSlots == 1 << 10, "the hash's shift");
    __syncthreads();
    const int m = nlisted, c = tid & (kLanes - 1);
    if (c >= C) return;
    for (int e = tid / kLanes; e < m; e += 256 / kLanes) {
        const int h = listed[e];
        float sum = 0.f;
        for (uint32_t p = head[h]; p != kNoPair; p = next[p]) {
            if constexpr (C > 1)
                sum += gs[(p >> 3) * C + c] * wgt[p];
            else
                sum += ORDER == 0 ? wgt[p] : g[p0 + (p >> 3)] * wgt[p];
        }
        if (sum != 0.f) atomicAdd(grad + (int64_t)key[h] * C + c, sum);
    }
}

// World to index coordinates (grid.py:77-78), a point to a thread, transposed to the
// rows that the gather and the scatter read.  As tensor operations this was five
// launches, 32 us of device time for 1.2M points and about as long on the host.
__global__ void __launch_bounds__(256) k_world_to_index(const float* __restrict__ pts, int64_t n,
                                                        const float* __restrict__ mn,
                                                        const float* __restrict__ mx,
                                                        const float* __restrict__ ws,
                                                        float* __restrict__ out) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
#pragma unroll
    for (int a = 0; a < 3; ++a) out[a * n + p] = (pts[3 * p + a] - mn[a]) / (mx[a] - mn[a]) * ws[a];
}

__device__ __forceinline__ bool slot_active(const TopoView& t, int64_t slot) {
    const int64_t leaf = slot >> 9;
    const int off = (int)(slot & 511);
    return (t.masks[leaf * 8 + (off >> 6)] >> (off & 63)) & 1ull;
}

__device__ __forceinline__ void slot_coord(const TopoView& t, int64_t slot, int& x, int& y,
                                           int& z) {
    const int64_t leaf = slot >> 9;
    const int off = (int)(slot & 511);
    x = t.origins[leaf * 3 + 0] + (off >> 6);
    y = t.origins[leaf * 3 + 1] + ((off >> 3) & 7);
    z = t.origins[leaf * 3 + 2] + (off & 7);
}

// copyFromDense (densityvdb.cu:31-48, colorvdb.cu:42-62): active slot <-
// dense[x][y][z][:] with z fastest.
__global__ void k_copy_from_dense(TopoView t, float* __restrict__ vals, int C,
                                  const float* __restrict__ dense, int rx, int ry, int rz) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= t.nleaf * 512) return;
    if (!slot_active(t, s)) return;
    int x, y, z;
    slot_coord(t, s, x, y, z);
    if (x < 0 || y < 0 || z < 0 || x >= rx || y >= ry || z >= rz) return;
    const float* src = dense + (((int64_t)x * ry + y) * rz + z) * C;
    for (int c = 0; c < C; ++c) vals[s * C + c] = src[c];
}

// Dense copy of the grid values over [0,rx)x[0,ry)x[0,rz): every voxel of an
// existing leaf (active or not) reads its stored value, others the background
// (OpenVDB tools::copyToDense semantics used by plenvdb.h:149-160,242-262).
__global__ void k_copy_to_dense(TopoView t, const float* __restrict__ vals, int C,
                                float* __restrict__ dense, int rx, int ry, int rz,
                                float background) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nvox = (int64_t)rx * ry * rz;
    if (q >= nvox) return;
    const int z = (int)(q % rz);
    const int y = (int)((q / rz) % ry);
    const int x = (int)(q / ((int64_t)ry * rz));
    const int64_t s = pvdb::slot_of(t, x, y, z);
    for (int c = 0; c < C; ++c) dense[q * C + c] = s >= 0 ? vals[s * C + c] : background;
}

// setValuesOn_bymask (densityvdb.cu:64-83): active slot <- val where mask.
__global__ void k_set_by_mask(TopoView t, float* __restrict__ vals,
                              const uint8_t* __restrict__ mask, float val, int rx, int ry,
                              int rz) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= t.nleaf * 512) return;
    if (!slot_active(t, s)) return;
    int x, y, z;
    slot_coord(t, s, x, y, z);
    if (x < 0 || y < 0 || z < 0 || x >= rx || y >= ry || z >= rz) return;
    if (mask[((int64_t)x * ry + y) * rz + z]) vals[s] = val;
}

// zero_grad (densityvdb.cu:353-361, colorvdb.cu:355-364): active slots only.
// One thread per V consecutive values of a slot, so that a wave's stores are
// contiguous: a thread per slot wrote its row in C stores 4 C bytes apart.  309k slots,
// 12 channels: 16.5 -> 5.9 us.
template <int V>
__global__ void __launch_bounds__(256) k_zero_active(TopoView t, float* __restrict__ grad, int C,
                                                     int64_t q0) {
    const int64_t q = q0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t s = q / (C / V);
    if (s >= t.nleaf * 512 || !slot_active(t, s)) return;
    if constexpr (V == 4)
        reinterpret_cast<float4*>(grad)[q] = make_float4(0.f, 0.f, 0.f, 0.f);
    else
        grad[q] = 0.f;
}

// Total-variation gradient of a VDB payload: the dense kernel's rule
// (total_variation_kernel.cu:13-35) on the grid's dense view over
// [0,rx)x[0,ry)x[0,rz) (stored value in an existing leaf, 0 elsewhere), applied
// to every slot inside that box.  Terms in the dense kernel's order z-1, z+1,
// y-1, y+1, x-1, x+1; the x axis takes wz, as there (lines 31-32).  One thread
// per (slot, V consecutive channels), so neighbouring threads read neighbouring
// 4V-byte pieces; a thread reads its own and its neighbours' values and writes
// only its own gradient, so no two threads touch one element.
//
// A workgroup lies within one leaf, so the leaf's origin and its six neighbours are
// the same for all its threads, and a thread's eight loads are issued together
// behind those two lookups: with lookups of its own at the leaf's faces, behind the
// gradient's load and branches, a thread made four round trips to memory in a row.
// 12 channels and one, twelve pairs of grids in turn: 600 leaves 25.5 -> 18.1 us, 1984
// leaves 65.4 -> 44.5.
//
// Without DENSE a voxel without a gradient is left alone, and costs its gradient's
// load only: that one is waited for first.  1984 leaves, 12 channels, gradients at
// all, 2% and none of the voxels: 50.5, 28.5 and 12.2 -> 37.6, 21.5 and 8.6 us (with
// the other loads ahead of the test 35.7, 26.0 and 21.1).
template <int V, bool DENSE>
__global__ void __launch_bounds__(256) k_tv_add_grad(TopoView t, const float* __restrict__ vals,
                                                     float* __restrict__ grad, int C, int rx,
                                                     int ry, int rz, float wy6, float wz6) {
    const int G = C / V;  // channel groups per slot
    // XCD-aware block order: workgroups are dealt to the 8 XCDs in turn, so
    // block b of the first 8*(n/8) is given the run (b % 8)*(n/8) + b/8 and each
    // XCD's L2 holds a contiguous range of slots with their in-leaf neighbours
    // (a bijection; the last n % 8 blocks keep their index)
    const unsigned nblk = gridDim.x, per = nblk / 8, bid = blockIdx.x;
    const unsigned lblk = bid < 8 * per ? (bid % 8) * per + bid / 8 : bid;
    const int64_t leaf = lblk / (2u * G);  // 512 G threads a leaf
    const unsigned in_leaf = (lblk - (unsigned)leaf * (2u * G)) * 256u + threadIdx.x;
    const int off = (int)(in_leaf / G), q = (int)(in_leaf - (unsigned)off * G);
    const int64_t s = leaf * 512 + off;
    using Vec = std::conditional_t<V == 4, float4, float>;
    auto ld = [&](const float* p, float* o) {
        const Vec w = *reinterpret_cast<const Vec*>(p);
        if constexpr (V == 4) {
            o[0] = w.x; o[1] = w.y; o[2] = w.z; o[3] = w.w;
        } else {
            o[0] = w;
        }
    };
    const int64_t e = s * C + (int64_t)q * V;
    float g0[V], v[V];
    ld(grad + e, g0);
    if constexpr (!DENSE) {
        bool any = false;
#pragma unroll
        for (int c = 0; c < V; ++c) any = any || g0[c] != 0.f;
        if (!any) return;
    }
    ld(vals + e, v);
    const int ox = t.origins[3 * leaf], oy = t.origins[3 * leaf + 1], oz = t.origins[3 * leaf + 2];
    const int32_t nl[6] = {pvdb::leaf_of(t, ox, oy, oz - 1), pvdb::leaf_of(t, ox, oy, oz + 8),
                           pvdb::leaf_of(t, ox, oy - 1, oz), pvdb::leaf_of(t, ox, oy + 8, oz),
                           pvdb::leaf_of(t, ox - 1, oy, oz), pvdb::leaf_of(t, ox + 8, oy, oz)};
    const int lx = off >> 6, ly = (off >> 3) & 7, lz = off & 7;
    const int x = ox + lx, y = oy + ly, z = oz + lz;
    if (x < 0 || y < 0 || z < 0 || x >= rx || y >= ry || z >= rz) return;
    // per direction: whether the neighbour lies in the box, on this leaf's far side, and
    // its offset from here in its leaf
    const bool in[6] = {z > 0, z < rz - 1, y > 0, y < ry - 1, x > 0, x < rx - 1};
    const bool out[6] = {lz == 0, lz == 7, ly == 0, ly == 7, lx == 0, lx == 7};
    const int step[3] = {1, 8, 64};
    const float w[6] = {wz6, wz6, wy6, wy6, wz6, wz6};
    float u[6][V], acc[V];
#pragma unroll
    for (int n = 0; n < 6; ++n) {  // a missing leaf's value is 0; this slot's stands in for the load
        const int d = step[n >> 1], sign = n & 1 ? 1 : -1;
        const int64_t at = !out[n] ? s + sign * d : nl[n] >= 0 ? (int64_t)nl[n] * 512 + off - sign * 7 * d : s;
        ld(vals + at * C + (int64_t)q * V, u[n]);
    }
#pragma unroll
    for (int c = 0; c < V; ++c) acc[c] = 0.f;
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        const bool missing = out[n] && nl[n] < 0;
#pragma unroll
        for (int c = 0; c < V; ++c) {
            const float term = w[n] * fminf(fmaxf(v[c] - (missing ? 0.f : u[n][c]), -1.f), 1.f);
            acc[c] = in[n] ? acc[c] + term : acc[c];
        }
    }
    float r[V];
#pragma unroll
    for (int c = 0; c < V; ++c) r[c] = (DENSE || g0[c] != 0.f) ? g0[c] + acc[c] : g0[c];
    if constexpr (V == 4)
        *reinterpret_cast<float4*>(grad + e) = make_float4(r[0], r[1], r[2], r[3]);
    else
        grad[e] = r[0];
}

__device__ __forceinline__ void adam1(float& p, float g, float& m, float& v, float sz, float eps,
                                      float b0, float b1) {
    const float nm = b0 * m + (1.f - b0) * g;
    const float nv = b1 * v + ((1.f - b1) * g) * g;
    m = nm;
    v = nv;
    p = p - (sz * nm) / (eps + sqrtf(nv));
}

// VDB Adam over all slots, one thread per (slot, group of `group` channels)
// (densityvdb.cu:185-349, colorvdb.cu:179-351).  G: the group, when it is known
// (0: any); a thread's loads are then all issued before its first store.  1M
// slots, 12 channels and one, 42% of the voxels updated, nothing cached: 84.9 ->
// 64.1 us for both grids.
template <int G>
__global__ void __launch_bounds__(256) k_vdb_adam(TopoView t, float* __restrict__ param,
                                                  const float* __restrict__ grad,
                                                  float* __restrict__ m, float* __restrict__ v,
                                                  const float* __restrict__ per_lr, int C,
                                                  int group, int mode, float stepsz, float eps,
                                                  float b0, float b1) {
    const int grp_n = G > 0 ? G : group;
    const int ngroups = C / grp_n;
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= t.nleaf * 512 * ngroups) return;
    const int64_t s = q / ngroups;
    const int64_t base = q * grp_n;
    if constexpr (G > 0) {
        float gg[G], pp[G], mm[G], vv[G];
#pragma unroll
        for (int c = 0; c < G; ++c) gg[c] = grad[base + c];
        if (!slot_active(t, s)) return;
        if (mode == 1) {
            bool all0 = true;
#pragma unroll
            for (int c = 0; c < G; ++c) all0 &= gg[c] == 0.f;
            if (all0) return;
        }
        const float sz = mode == 2 ? per_lr[s] * stepsz : stepsz;
#pragma unroll
        for (int c = 0; c < G; ++c) {
            mm[c] = m[base + c];
            vv[c] = v[base + c];
            pp[c] = param[base + c];
        }
#pragma unroll
        for (int c = 0; c < G; ++c) {
            adam1(pp[c], gg[c], mm[c], vv[c], sz, eps, b0, b1);
            m[base + c] = mm[c];
            v[base + c] = vv[c];
            param[base + c] = pp[c];
        }
    } else {
        if (!slot_active(t, s)) return;
        if (mode == 1) {
            bool all0 = true;
            for (int c = 0; c < group; ++c) all0 &= grad[base + c] == 0.f;
            if (all0) return;
        }
        const float sz = mode == 2 ? per_lr[s] * stepsz : stepsz;
        for (int c = 0; c < group; ++c)
            adam1(param[base + c], grad[base + c], m[base + c], v[base + c], sz, eps, b0, b1);
    }
}

// Dense Adam (plenvdb/lib/cuda/adam_upd_kernel.cu:8-58).
__global__ void k_dense_adam(float* __restrict__ p, const float* __restrict__ g,
                             float* __restrict__ m, float* __restrict__ v,
                             const float* __restrict__ per_lr, int64_t n, int mode,
                             float step_size, float eps, float b0, float b1) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const float gg = g[q];
    if (mode == 1 && gg == 0.f) return;
    const float nm = b0 * m[q] + (1.f - b0) * gg;
    const float nv = b1 * v[q] + ((1.f - b1) * gg) * gg;
    m[q] = nm;
    v[q] = nv;
    float sz = step_size;
    if (mode == 2) sz = sz * per_lr[q];
    p[q] = p[q] - (sz * nm) / (sqrtf(nv) + eps);
}

template <int C, int ORDER>
void launch_fwd(const TopoView& t, const float* vals, int cdyn, const float* xs, const float* ys,
                const float* zs, int64_t n, float* out, hipStream_t s) {
    hipLaunchKernelGGL((k_tri_fwd<C, ORDER>), dim3(pvdb_blocks(n, 256)), dim3(256), 0, s, t, vals,
                       cdyn, xs, ys, zs, n, out, reinterpret_cast<uintptr_t>(vals) % 16 == 0);
}
template <int C, int ORDER>
void launch_bwd(const TopoView& t, float* grad, int cdyn, const float* xs, const float* ys,
                const float* zs, const float* g, int64_t n, hipStream_t s) {
    if constexpr (C > 0) {
        if (t.nleaf < (int64_t(1) << 23) - 1) {  // every slot below the hash's empty key
            const int64_t most = pvdb_launch_items(kBwdPoints, 256);
            for (int64_t p = 0; p < n; p += most) {
                const int64_t m = n - p < most ? n - p : most;
                hipLaunchKernelGGL((k_tri_bwd_agg<C, ORDER>), dim3(pvdb_blocks(m, kBwdPoints)),
                                   dim3(256), 0, s, t, grad, xs + p, ys + p, zs + p, g + C * p, m);
            }
            return;
        }
    }
    hipLaunchKernelGGL((k_tri_bwd<C, ORDER>), dim3(pvdb_blocks(n, 256)), dim3(256), 0, s, t, grad,
                       cdyn, xs, ys, zs, g, n);
}

int check_topo(const pvdb_topology* t) {
    if (!t) {
        pvdb::set_error("null topology");
        return PVDB_EHANDLE;
    }
    return PVDB_OK;
}

}  // namespace

extern "C" {

int pvdb_trilinear_fwd(const pvdb_topology* topo, const float* vals, int32_t channels,
                       int32_t order, const float* xs, const float* ys, const float* zs,
                       int64_t n, float* out, void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && channels <= 48, "channels must be in [1, 48]");
    PVDB_CHECK_ARG(order == 0 || order == 1, "order must be 0 (density) or 1 (color)");
    PVDB_CHECK_ARG(order == 1 || channels == 1, "density order needs one channel");
    PVDB_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return PVDB_OK;
    PVDB_CHECK_ARG(vals && xs && ys && zs && out, "null pointer");
    const TopoView t = pvdb::view_of(topo);
    hipStream_t s = (hipStream_t)stream;
    if (order == 0)
        launch_fwd<1, 0>(t, vals, 1, xs, ys, zs, n, out, s);
    else if (channels == 1)
        launch_fwd<1, 1>(t, vals, 1, xs, ys, zs, n, out, s);
    else if (channels == 3)
        launch_fwd<3, 1>(t, vals, 3, xs, ys, zs, n, out, s);
    else if (channels == 12)
        launch_fwd<12, 1>(t, vals, 12, xs, ys, zs, n, out, s);
    else
        launch_fwd<0, 1>(t, vals, channels, xs, ys, zs, n, out, s);
    PVDB_LAUNCHED("k_tri_fwd");
    return PVDB_OK;
}

int pvdb_trilinear_bwd(const pvdb_topology* topo, float* grad, int32_t channels, int32_t order,
                       const float* xs, const float* ys, const float* zs, const float* g,
                       int64_t n, void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && channels <= 48, "channels must be in [1, 48]");
    PVDB_CHECK_ARG(order == 0 || order == 1, "order must be 0 (density) or 1 (color)");
    PVDB_CHECK_ARG(order == 1 || channels == 1, "density order needs one channel");
    PVDB_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return PVDB_OK;
    PVDB_CHECK_ARG(grad && xs && ys && zs && g, "null pointer");
    const TopoView t = pvdb::view_of(topo);
    hipStream_t s = (hipStream_t)stream;
    if (order == 0)
        launch_bwd<1, 0>(t, grad, 1, xs, ys, zs, g, n, s);
    else if (channels == 1)
        launch_bwd<1, 1>(t, grad, 1, xs, ys, zs, g, n, s);
    else if (channels == 3)
        launch_bwd<3, 1>(t, grad, 3, xs, ys, zs, g, n, s);
    else if (channels == 12)
        launch_bwd<12, 1>(t, grad, 12, xs, ys, zs, g, n, s);
    else
        launch_bwd<0, 1>(t, grad, channels, xs, ys, zs, g, n, s);
    PVDB_LAUNCHED("k_tri_bwd");
    return PVDB_OK;
}

int pvdb_copy_from_dense(const pvdb_topology* topo, float* vals, int32_t channels,
                         const float* dense, int32_t rx, int32_t ry, int32_t rz, void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && rx > 0 && ry > 0 && rz > 0, "bad sizes");
    PVDB_CHECK_ARG(vals && dense, "null pointer");
    const TopoView t = pvdb::view_of(topo);
    if (t.nleaf == 0) return PVDB_OK;
    hipLaunchKernelGGL(k_copy_from_dense, dim3(pvdb_blocks(t.nleaf * 512, 256)), dim3(256), 0,
                       (hipStream_t)stream, t, vals, channels, dense, rx, ry, rz);
    PVDB_LAUNCHED("k_copy_from_dense");
    return PVDB_OK;
}

int pvdb_copy_to_dense(const pvdb_topology* topo, const float* vals, int32_t channels,
                       float* dense, int32_t rx, int32_t ry, int32_t rz, float background,
                       void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && rx > 0 && ry > 0 && rz > 0, "bad sizes");
    PVDB_CHECK_ARG(vals && dense, "null pointer");
    const TopoView t = pvdb::view_of(topo);
    const int64_t nvox = (int64_t)rx * ry * rz;
    hipLaunchKernelGGL(k_copy_to_dense, dim3(pvdb_blocks(nvox, 256)), dim3(256), 0,
                       (hipStream_t)stream, t, vals, channels, dense, rx, ry, rz, background);
    PVDB_LAUNCHED("k_copy_to_dense");
    return PVDB_OK;
}

int pvdb_set_values_by_mask(const pvdb_topology* topo, float* vals, const uint8_t* mask,
                            float value, int32_t rx, int32_t ry, int32_t rz, void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(rx > 0 && ry > 0 && rz > 0, "bad sizes");
    PVDB_CHECK_ARG(vals && mask, "null pointer");
    const TopoView t = pvdb::view_of(topo);
    if (t.nleaf == 0) return PVDB_OK;
    hipLaunchKernelGGL(k_set_by_mask, dim3(pvdb_blocks(t.nleaf * 512, 256)), dim3(256), 0,
                       (hipStream_t)stream, t, vals, mask, value, rx, ry, rz);
    PVDB_LAUNCHED("k_set_by_mask");
    return PVDB_OK;
}

int pvdb_tv_add_grad(const pvdb_topology* topo, const float* vals, float* grad,
                     int32_t channels, int32_t rx, int32_t ry, int32_t rz, float wx, float wy,
                     float wz, int32_t dense_mode, void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && rx > 0 && ry > 0 && rz > 0, "bad sizes");
    PVDB_CHECK_ARG(vals && grad, "null pointer");
    (void)wx;  // the dense kernel weighs the x axis with wz
    const TopoView t = pvdb::view_of(topo);
    if (t.nleaf == 0) return PVDB_OK;
    // weights scaled on the host as total_variation_kernel.cu:45-47 does; four
    // channels per thread when the row splits into 16-byte pieces
    const bool vec4 = channels % 4 == 0 && reinterpret_cast<uintptr_t>(vals) % 16 == 0 &&
                      reinterpret_cast<uintptr_t>(grad) % 16 == 0;
    const int64_t nthreads = t.nleaf * 512 * (vec4 ? channels / 4 : channels);
    const auto kernel = dense_mode ? (vec4 ? k_tv_add_grad<4, true> : k_tv_add_grad<1, true>)
                                   : (vec4 ? k_tv_add_grad<4, false> : k_tv_add_grad<1, false>);
    hipLaunchKernelGGL(kernel, dim3(pvdb_blocks(nthreads, 256)), dim3(256), 0, (hipStream_t)stream,
                       t, vals, grad, channels, rx, ry, rz, wy / 6.f, wz / 6.f);
    PVDB_LAUNCHED("k_tv_add_grad");
    return PVDB_OK;
}

int pvdb_world_to_index(const float* pts, int64_t n, const float* xyz_min, const float* xyz_max,
                        const float* ws_minus_1, float* out, void* stream) {
    PVDB_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return PVDB_OK;
    PVDB_CHECK_ARG(pts && xyz_min && xyz_max && ws_minus_1 && out, "null pointer");
    hipLaunchKernelGGL(k_world_to_index, dim3(pvdb_blocks(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, pts, n, xyz_min, xyz_max, ws_minus_1, out);
    PVDB_LAUNCHED("k_world_to_index");
    return PVDB_OK;
}

int pvdb_zero_active(const pvdb_topology* topo, float* grad, int32_t channels, void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && grad, "bad arguments");
    const TopoView t = pvdb::view_of(topo);
    if (t.nleaf == 0) return PVDB_OK;
    const bool vec4 = channels % 4 == 0 && reinterpret_cast<uintptr_t>(grad) % 16 == 0;
    const int64_t n = t.nleaf * 512 * (vec4 ? channels / 4 : channels);
    const int64_t most = pvdb_launch_items(256, 256);
    for (int64_t q = 0; q < n; q += most) {
        const int64_t m = n - q < most ? n - q : most;
        hipLaunchKernelGGL(vec4 ? k_zero_active<4> : k_zero_active<1>, dim3(pvdb_blocks(m, 256)),
                           dim3(256), 0, (hipStream_t)stream, t, grad, channels, q);
        PVDB_LAUNCHED("k_zero_active");
    }
    return PVDB_OK;
}

int pvdb_vdb_adam(const pvdb_topology* topo, float* param, const float* grad, float* exp_avg,
                  float* exp_avg_sq, const float* per_lr, int32_t channels, int32_t group,
                  int32_t mode, float stepsz, float eps, float beta0, float beta1,
                  void* stream) {
    if (int rc = check_topo(topo)) return rc;
    PVDB_CHECK_ARG(channels >= 1 && group >= 1 && channels % group == 0, "bad channel grouping");
    PVDB_CHECK_ARG(mode >= 0 && mode <= 2, "mode must be 0, 1 or 2");
    PVDB_CHECK_ARG(mode != 2 || per_lr, "mode 2 needs per-voxel lr");
    PVDB_CHECK_ARG(param && grad && exp_avg && exp_avg_sq, "null pointer");
    const TopoView t = pvdb::view_of(topo);
    if (t.nleaf == 0) return PVDB_OK;
    const int64_t n = t.nleaf * 512 * (channels / group);
    const auto kernel = group == 3 ? k_vdb_adam<3> : group == 1 ? k_vdb_adam<1> : k_vdb_adam<0>;
    hipLaunchKernelGGL(kernel, dim3(pvdb_blocks(n, 256)), dim3(256), 0, (hipStream_t)stream,
                       t, param, grad, exp_avg, exp_avg_sq, per_lr, channels, group, mode, stepsz,
                       eps, beta0, beta1);
    PVDB_LAUNCHED("k_vdb_adam");
    return PVDB_OK;
}

int pvdb_dense_adam(float* param, const float* grad, float* exp_avg, float* exp_avg_sq,
                    const float* per_lr, int64_t n, int32_t mode, float step_size, float eps,
                    float beta0, float beta1, void* stream) {
    PVDB_CHECK_ARG(n >= 0, "n must be >= 0");
    PVDB_CHECK_ARG(mode >= 0 && mode <= 2, "mode must be 0, 1 or 2");
    PVDB_CHECK_ARG(mode != 2 || per_lr, "mode 2 needs per-element lr");
    if (n == 0) return PVDB_OK;
    PVDB_CHECK_ARG(param && grad && exp_avg && exp_avg_sq, "null pointer");
    hipLaunchKernelGGL(k_dense_adam, dim3(pvdb_blocks(n, 256)), dim3(256), 0, (hipStream_t)stream,
                       param, grad, exp_avg, exp_avg_sq, per_lr, n, mode, step_size, eps, beta0,
                       beta1);
    PVDB_LAUNCHED("k_dense_adam");
    return PVDB_OK;
}

}  // extern "C"
