// Fused step: the grid gradients of large batches, by cell.
//
// k_scatter_agg (fused_scatter.hip) adds a slot's 13 sums once per chunk of 64
// records, about a ray's piece, and is bound by those atomics: they execute past
// the L2 caches, a value at a time (200G a second), 2.8 rows of 13 a record
// whatever the batch.  When a batch puts thousands of records into a leaf, their
// cells and corners coincide.  Here the record numbers are ordered by cell, and a
// workgroup sums a leaf's cells in LDS over the 10 x 10 x 10 voxels that they can
// touch, and adds each voxel's row to the grids once.
//
//   k_cell_count  a record's cell (of the leaf of its nearest voxel) and its rank there
//   k_cell_scan   per leaf, the cells' counts as an exclusive prefix, and the total
//   k_leaf_scan   the leaves' starts, and the parts of leaves with many records
//   k_cell_order  record numbers to their places
//   k_cell_sums   the sums.  LDS float atomics take 180 cycles a wavefront (plain LDS
//                 accesses below 20), so there are none: a cell's eight corner rows
//                 are summed in registers by 16 lanes, a channel each, and cells of
//                 the same parity on each axis share no corner, so eight passes with a
//                 barrier between them add them up with plain reads and writes.
//
// 7.80M records in 1984 leaves: 1400 us by chunks, 713 us by cells, of which the
// sums are 438 (bound by the latency of the records' 64-byte rows, read in the
// cells' order, four ahead a lane group), the counts 161 (returning atomics, one for
// a run of a ray's samples in a cell: one for each took 245) and the order 93.
#include "fused_common.h"
#include "gather.h"
#include "plenvdb_hip.h"

using namespace pvdb;

namespace {

constexpr int kSide = 10, kBox = kSide * kSide * kSide;  // voxels -1 .. 8 from the leaf's origin
constexpr int kRow = 13;                                 // 12 colour gradients, dL/dsigma
constexpr int kSig = kSigmaAt<12>;

// A record whose nearest voxel's leaf is missing (the march kept it by a rounding of
// its own): its corners' values straight to the grids.
__device__ void add_record(const TopoView& t, const float4& p, uint32_t bits, const float* g,
                           const GradRows& G, uint8_t* leaf_touched) {
    const Cell cell = make_cell(p.x, p.y, p.z);
    for (int q = 0; q < 8; ++q) {
        const int dx = (kCx >> q) & 1, dy = (kCy >> q) & 1, dz = (kCz >> q) & 1;
        const int i = cell.i0 + dx, j = cell.j0 + dy, k = cell.k0 + dz;
        const int32_t leaf = leaf_of(t, i, j, k);
        if (leaf < 0) continue;
        const float w = ((dx ? cell.u : 1.f - cell.u) * (dy ? cell.v : 1.f - cell.v)) *
                        (dz ? cell.w : 1.f - cell.w);
        const int64_t s = (int64_t)leaf * 512 + voxel_offset(i, j, k);
        leaf_touched[leaf] = 1;
        if (bits & kAliveA) atomicAdd(G.density + s * G.ds, g[kSig] * w);
        if (bits & kAliveW)
            for (int c = 0; c < 12; ++c) atomicAdd(G.color + s * G.cs + c, g[c] * w);
    }
}

__global__ void __launch_bounds__(256) k_cell_clear(CellBins B, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) B.count[i] = 0;
}

// The first workgroups sum the MLP's dW partials and the loss (as in k_scatter_agg's
// launch).
__global__ void __launch_bounds__(256) k_cell_count(TopoView t, RayBuffers R, Records rec,
                                                    int64_t capacity, CellBins B, GradRows G,
                                                    uint8_t* __restrict__ leaf_touched,
                                                    ReduceArgs red) {
    __shared__ float4 scratch[kReduceGrp * kReduceVec];
    if ((int)blockIdx.x < red.blocks) {  // uniform over the workgroup
        dw_reduce_block(blockIdx.x, red.part, red.nparts, red.dw, red.adam, scratch);
        return;
    }
    const int lead = red.blocks + (red.ray_loss ? 1 : 0);
    if ((int)blockIdx.x < lead) {
        if (threadIdx.x < 64) loss_sum_wave(red.ray_loss, red.n_rays, red.loss);
        return;
    }
    const int64_t total = min((int64_t)R.total[0], capacity);
    const int64_t step = (int64_t)(gridDim.x - lead) * 256;
    const int lane = lane_id();
    for (int64_t q0 = (int64_t)(blockIdx.x - lead) * 256 + (threadIdx.x & ~63); q0 < total; q0 += step) {
        const int64_t q = q0 + lane;
        const uint32_t bits = q < total ? __float_as_uint(rec.ab[q].y) : 0u;
        int cell = -1;
        if (bits & (kAliveA | kAliveW)) {
            const float4 p = rec.xyze[q];
            const int v[3] = {(int)floorf(p.x + 0.5f), (int)floorf(p.y + 0.5f), (int)floorf(p.z + 0.5f)};
            const int32_t leaf = leaf_of(t, v[0], v[1], v[2]);
            if (leaf < 0) {
                add_record(t, p, bits, reinterpret_cast<const float*>(rec.grad + 4 * q), G, leaf_touched);
            } else {
                // lower corners -1 .. 7 from the leaf's origin: the nearest voxel is the
                // lower corner or the one after it on each axis
                const int x = (int)floorf(p.x) + 1 - (v[0] & ~7), y = (int)floorf(p.y) + 1 - (v[1] & ~7),
                          z = (int)floorf(p.z) + 1 - (v[2] & ~7);
                cell = leaf * kLeafCells + (x * kCellSide + y) * kCellSide + z;
            }
        }
        // one atomic for a run of lanes in the same cell (a ray's samples, half a voxel apart)
        const int before = __shfl_up(cell, 1, 64);
        const uint64_t heads = __ballot(lane == 0 || cell != before), upto = ~0ull >> (63 - lane);
        const int head = 63 - __clzll((long long)(heads & upto));
        const uint64_t past = heads & ~upto;
        int rank = 0;
        if (head == lane && cell >= 0)
            rank = atomicAdd(B.count + cell,
                             (past ? __ffsll((unsigned long long)past) - 1 : 64) - lane);
        rank = __shfl(rank, head, 64) + (lane - head);
        if (q < total) B.at[q] = make_int2(cell, rank);
    }
}

// A workgroup per leaf: counts to exclusive prefixes, in place.
__global__ void __launch_bounds__(256) k_cell_scan(CellBins B) {
    static_assert(kLeafCells <= 3 * 256, "three counts to a thread");
    __shared__ int wsum[4];
    int32_t* const c = B.count + (int64_t)blockIdx.x * kLeafCells;
    const int tid = threadIdx.x, lane = tid & 63;
    int v[3], sum = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        v[k] = 3 * tid + k < kLeafCells ? c[3 * tid + k] : 0;
        sum += v[k];
    }
    int inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(inc, d, 64);
        if (lane >= d) inc += o;
    }
    if (lane == 63) wsum[tid >> 6] = inc;
    __syncthreads();
    int run = inc - sum;
    for (int w = 0; w < (tid >> 6); ++w) run += wsum[w];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (3 * tid + k < kLeafCells) c[3 * tid + k] = run;
        run += v[k];
    }
    if (tid == 255) B.leaf[blockIdx.x] = run;
}

// The leaves' totals to starts (start[nleaf]: all), and the leaves' parts: one
// workgroup.
__global__ void __launch_bounds__(1024) k_leaf_scan(CellBins B, RayBuffers R, int64_t capacity,
                                                    int nleaf) {
    __shared__ int wsum[16], psum[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    // about 1024 parts in all: fewer leave CUs idle, and each adds up to 1000 rows (more
    // of them above 8.4M records, at 8192 a part)
    const int total = (int)min((int64_t)R.total[0], capacity);
    const int per = min(max(total / 1024, kMinPart), 8 * kMinPart);
    int carry = 0, parts0 = 0;  // below 2^31: the capacity is
    for (int b0 = 0; b0 < nleaf; b0 += 1024) {
        const int b = b0 + tid, n = b < nleaf ? B.leaf[b] : 0;
        const int parts = n / per + (n % per ? 1 : 0);
        int inc = n, pinc = parts;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d, 64), po = __shfl_up(pinc, d, 64);
            if (lane >= d) {
                inc += o;
                pinc += po;
            }
        }
        if (lane == 63) {
            wsum[wv] = inc;
            psum[wv] = pinc;
        }
        __syncthreads();
        int before = carry, pbefore = parts0;
        for (int w = 0; w < 16; ++w) {
            if (w < wv) {
                before += wsum[w];
                pbefore += psum[w];
            }
            carry += wsum[w];
            parts0 += psum[w];
        }
        if (b < nleaf) {
            B.leaf[b] = before + inc - n;
            for (int k = 0; k < parts; ++k) B.part[pbefore + pinc - parts + k] = make_int4(b, k, parts, 0);
        }
        __syncthreads();  // wsum and psum are reused
    }
    if (tid == 0) {
        B.leaf[nleaf] = carry;
        B.nparts[0] = parts0;
    }
}

__global__ void __launch_bounds__(256) k_cell_order(RayBuffers R, int64_t capacity, CellBins B) {
    const int64_t total = min((int64_t)R.total[0], capacity);
    const int64_t step = (int64_t)gridDim.x * 256;
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < total; q += step) {
        const int2 at = B.at[q];
        if (at.x >= 0) B.order[B.leaf[at.x / kLeafCells] + B.count[at.x] + at.y] = (int32_t)q;
    }
}

constexpr int kCellThreads = 512, kGroups = kCellThreads / 16;
constexpr int kAhead = 4;  // records of a lane group whose loads are in flight
__global__ void __launch_bounds__(kCellThreads, 6) k_cell_sums(TopoView t, Records rec, CellBins B,
                                                               GradRows G,
                                                               uint8_t* __restrict__ leaf_touched) {
    __shared__ float acc[kBox * kRow];
    __shared__ int32_t near_leaf[27];
    const int tid = threadIdx.x, lane = lane_id(), c = tid & 15, grp = tid >> 4;
    const float* const grad = reinterpret_cast<const float*>(rec.grad) + (c < 12 ? c : kSig);
    const int nparts = B.nparts[0];
    for (int part = blockIdx.x; part < nparts; part += gridDim.x) {
        // the part's share of each cell's records; parts of a leaf come next to each other
        const int4 pt = B.part[part];
        const int l = pt.x;
        const int32_t* const cells = B.count + (int64_t)l * kLeafCells;
        const int start = B.leaf[l], all = B.leaf[l + 1] - start;
        const int o0 = t.origins[3 * (int64_t)l] - 1, o1 = t.origins[3 * (int64_t)l + 1] - 1,
                  o2 = t.origins[3 * (int64_t)l + 2] - 1;  // the box's first voxel
        for (int e = tid; e < kBox * kRow; e += kCellThreads) acc[e] = 0.f;
        if (tid < 27)
            near_leaf[tid] = leaf_of(t, o0 + 1 + 8 * (tid / 9 - 1), o1 + 1 + 8 * ((tid / 3) % 3 - 1),
                                     o2 + 1 + 8 * (tid % 3 - 1));
        __syncthreads();
        for (int pass = 0; pass < 8; ++pass) {
            const int px = pass >> 2, py = (pass >> 1) & 1, pz = pass & 1;  // the cells' parities
            const int ny = 5 - py, nz = 5 - pz, ncell = (5 - px) * ny * nz;
            // the group's cells grp, grp + kGroups, ...: lane k holds the k-th one's
            static_assert(125 <= 16 * kGroups, "a lane to each of the group's cells");
            int cell = -1, first = 0, count = 0;
            if (grp + kGroups * c < ncell) {
                const int e = grp + kGroups * c;
                cell = ((2 * (e / (ny * nz)) + px) * kCellSide + 2 * ((e / nz) % ny) + py) * kCellSide +
                       2 * (e % nz) + pz;
                first = cells[cell];
                count = (cell + 1 < kLeafCells ? cells[cell + 1] : all) - first;
                const int p0 = (int)((int64_t)count * pt.y / pt.z);
                count = (int)((int64_t)count * (pt.y + 1) / pt.z) - p0;
                first += p0;
            }
            for (int k = 0; grp + kGroups * k < ncell; ++k) {  // uniform over the lane group
                const int src = (lane & 48) | k;
                const int n = __shfl(count, src, 64), f = start + __shfl(first, src, 64),
                          ce = __shfl(cell, src, 64);
                if (n == 0) continue;
                float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                for (int r0 = 0; r0 < n; r0 += 16) {
                    const int mine = r0 + c < n ? B.order[f + r0 + c] : 0;
                    const int m = min(16, n - r0);
                    auto number = [&](int i) { return __shfl(mine, (lane & 48) | min(i, m - 1), 64); };
                    float4 p[kAhead];
                    float g[kAhead];
                    auto load = [&](int i, int k) {
                        const int q = number(i);
                        p[k] = rec.xyze[q];
                        g[k] = grad[16 * (int64_t)q];
                    };
                    auto add = [&](int k) {
                        const Cell w = make_cell(p[k].x, p[k].y, p[k].z);
                        // corner 4 dx + 2 dy + dz; a row's colours are zero unless the record
                        // is weight-kept, its dL/dsigma unless it is alpha-kept
                        const float x1 = g[k] * w.u, x0 = g[k] * (1.f - w.u), v0 = 1.f - w.v,
                                    w0 = 1.f - w.w;
                        const float y[4] = {x0 * v0, x0 * w.v, x1 * v0, x1 * w.v};
#pragma unroll
                        for (int h = 0; h < 4; ++h) {
                            s[2 * h] += y[h] * w0;
                            s[2 * h + 1] += y[h] * w.w;
                        }
                    };
#pragma unroll
                    for (int k = 0; k < kAhead; ++k) load(k, k);  // the last one again past the end
                    int i = 0;
                    for (; i + kAhead <= m; i += kAhead)
#pragma unroll
                        for (int k = 0; k < kAhead; ++k) {
                            add(k);
                            load(i + kAhead + k, k);
                        }
#pragma unroll
                    for (int k = 0; k < kAhead; ++k)
                        if (i + k < m) add(k);
                }
                if (c < kRow) {
                    const int x = ce / (kCellSide * kCellSide), y = (ce / kCellSide) % kCellSide,
                              z = ce % kCellSide;
                    float* a = acc + ((x * kSide + y) * kSide + z) * kRow + c;
#pragma unroll
                    for (int h = 0; h < 8; ++h)
                        a[(((h >> 2) * kSide + ((h >> 1) & 1)) * kSide + (h & 1)) * kRow] += s[h];
                }
            }
            __syncthreads();
        }
        for (int r = grp; r < kBox; r += kGroups) {
            const int x = r / (kSide * kSide), y = (r / kSide) % kSide, z = r % kSide;
            const float s = c < kRow ? acc[r * kRow + c] : 0.f;
            const uint32_t any = (uint32_t)(__ballot(s != 0.f) >> (lane & 48)) & 0xffffu;
            const int32_t leaf = near_leaf[(((x + 7) >> 3) * 3 + ((y + 7) >> 3)) * 3 + ((z + 7) >> 3)];
            if (!any || leaf < 0) continue;
            const int64_t slot = (int64_t)leaf * 512 + voxel_offset(o0 + x, o1 + y, o2 + z);
            if (s != 0.f)  // adding zero changes nothing
                atomicAdd(c < 12 ? G.color + slot * G.cs + c : G.density + slot * G.ds, s);
            if (c == 13) leaf_touched[leaf] = 1;
        }
        __syncthreads();  // acc and near_leaf are reused
    }
}

}  // namespace

namespace pvdb {

int launch_scatter_cells(const TopoView& t, const RayBuffers& R, const Records& rec, int64_t capacity,
                         const CellBins& B, const GradRows& G, uint8_t* leaf_touched,
                         const ReduceArgs& red, hipStream_t s) {
    constexpr int kGrid = 2048;  // persistent: the record count stays on the device
    const int lead = red.blocks + (red.ray_loss ? 1 : 0);
    const int64_t ncell = t.nleaf * kLeafCells;
    hipLaunchKernelGGL(k_cell_clear, dim3(pvdb_blocks(ncell, 256)), dim3(256), 0, s, B, ncell);
    PVDB_LAUNCHED("k_cell_clear");
    hipLaunchKernelGGL(k_cell_count, dim3(kGrid + lead), dim3(256), 0, s, t, R, rec, capacity, B, G,
                       leaf_touched, red);
    PVDB_LAUNCHED("k_cell_count");
    hipLaunchKernelGGL(k_cell_scan, dim3((unsigned)t.nleaf), dim3(256), 0, s, B);
    PVDB_LAUNCHED("k_cell_scan");
    hipLaunchKernelGGL(k_leaf_scan, dim3(1), dim3(1024), 0, s, B, R, capacity, (int)t.nleaf);
    PVDB_LAUNCHED("k_leaf_scan");
    hipLaunchKernelGGL(k_cell_order, dim3(kGrid), dim3(256), 0, s, R, capacity, B);
    PVDB_LAUNCHED("k_cell_order");
    // three workgroups a CU by LDS, taking parts in turn
    hipLaunchKernelGGL(k_cell_sums, dim3(768), dim3(kCellThreads), 0, s, t, rec, B, G, leaf_touched);
    PVDB_LAUNCHED("k_cell_sums");
    return PVDB_OK;
}

}  // namespace pvdb
