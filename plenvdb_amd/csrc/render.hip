// Merged-VDB renderer: MGRenderer::render_an_image (plenvdb/lib/vdb/plenvdb.h:
// 1029-1035 -> renderer.cu:370-424) in four kernels and no host round trip.
//
// The reference renders in two full marches per pixel (first_look_merged
// counts the kept samples and rewrites t_min / t_max, renderer.cu:222-268;
// ray_marching_merged re-marches from the rewritten t_min and gathers them,
// :312-367), a host read-back of the sample total, four SGEMMs over the
// materialised sample list (cuda_rgbnet, :83-109) and an atomic composite
// (final_render, :112-119).  Here:
//
//   k_render_count  the first march with trigetDensity's summation order, L
//                   lanes per pixel taking L consecutive steps at a time (a
//                   wave per block of 64 / L pixels); stores the kept count and
//                   the rewritten (t_min, t_max) per pixel.
//   k_render_fill   the second march from the rewritten t_min with
//                   trigetDensity2's order: the tile reserves its records with
//                   one atomic (counts scanned across the wave) and writes one
//                   32-byte record per kept sample (its cell, fractions,
//                   weight and pixel), at most the first march's count of
//                   them, contiguous per pixel.  So the sample set is the
//                   reference's, including the second march's restart
//                   (renderer.cu:263).
//   k_render_mlp    persistent waves over 32-record groups: the records' colour
//                   features gathered under the group before's MFMAs, the RGB MLP on
//                   v_mfma_f32_32x32x16_f16 (weights in LDS) and each record's
//                   contribution w / (1 + exp(-raw)) (final_render).
//   k_render_composite  per pixel: T_last * bg plus its records' contributions,
//                   eight lanes per pixel reading its run of records together
//                   (a fixed order, so frames are reproducible).
//
// Data layout.  The merged index grid (vdb_compression.py:19-59: index 1 +
// rank of an active voxel, 0 elsewhere) is a topology whose value masks are
// the non-zero indices, plus a slot-major payload holding, per slot, density
// and the 12 colour channels of the voxel's index (index 0's values for
// inactive voxels; slot `nslots` holds index 0's values for corners whose leaf
// does not exist).  A slot is 32 bytes (fp16: exact for the fp16 data of
// mergeddata.npz) or 64 bytes (fp32); the leaves' density cells follow
// (k_render_cells), which the marches read.
//
// MLP.  Layer outputs are computed transposed (features x samples) and stay in
// registers: the D fragment of one layer is the B fragment of the next once the
// next layer's weights are stored with their K index permuted accordingly (see
// rperm).  Weights are fp16 in LDS, read as 16-byte fragments.  The first layer's
// input row is [feature 0..11 | PE 0..26 | 1] (40 halves), so its bias is a weight
// column; a pixel's PE row holds column c at position c - 8.
#include <cmath>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "gather.h"
#include "mfma_util.h"
#include "plenvdb_hip.h"
#include "pvdb_common.h"

namespace pvdb {
TopoView view_of(const pvdb_topology* t);
}

using namespace pvdb;

namespace {

constexpr int kHid = 128;
constexpr int kMlpWaves = 4;  // MLP waves per workgroup: they share the LDS weights
// The MLP's LDS image, as pvdb_render_pack_weights lays it out.
struct alignas(16) RenderSmem {
    uint4 w0[6 * 128];  // [chunk][hidden feature]: W0^T columns 8c .. 8c + 7 (39: b0; 40..47: 0)
    uint4 w1[32 * 64];  // [row tile][k-step][lane]: W1^T's A fragments, K permuted
    uint4 w2[8 * 2 * 4];  // [k-step][h][logit]: W2^T rows, K permuted
    float b[128 + 4];   // b1, b2
};
constexpr int kW0Frag = 6 * 128 * 8, kW1Frag = 32 * 64 * 8, kW2Frag = 8 * 2 * 4 * 8;
constexpr int kPackedHalves = kW0Frag + kW1Frag + kW2Frag;
constexpr int kBiasFloats = 128 + 4;
constexpr int kPackedBytes = kPackedHalves * 2 + kBiasFloats * 4;
static_assert(sizeof(RenderSmem) == kPackedBytes, "the image is the struct");
constexpr int kMarchThreads = 256;    // 4 waves per march workgroup
constexpr int64_t kMaxRecords = 0x7fffffffll;  // record indices are int32 in the pixel table

// Position j (0..7) of k-step s in lane half h holds feature rperm(s, h, j): what
// that half of the previous layer's D fragments carries.
__host__ __device__ __forceinline__ int rperm(int s, int h, int j) {
    return 16 * s + 8 * (j >> 2) + 4 * h + (j & 3);
}

__global__ void k_render_pack(const float* __restrict__ w0, const float* __restrict__ b0,
                              const float* __restrict__ w1, const float* __restrict__ b1,
                              const float* __restrict__ w2, const float* __restrict__ b2,
                              int dcol, int dpe, int dout, _Float16* __restrict__ outh,
                              float* __restrict__ outb) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < kW0Frag) {
        const int in = 8 * (idx >> 10) + (idx & 7), o = (idx >> 3) & 127;
        outh[idx] = (_Float16)(in < dcol + dpe ? w0[in * kHid + o] : in == dcol + dpe ? b0[o] : 0.f);
    } else if (idx < kW0Frag + kW1Frag) {
        const int q = idx - kW0Frag;
        const int lane = (q >> 3) & 63, ts = q >> 9;
        outh[idx] = (_Float16)w1[rperm(ts & 7, lane >> 5, q & 7) * kHid + 32 * (ts >> 3) + (lane & 31)];
    } else if (idx < kPackedHalves) {
        const int q = idx - kW0Frag - kW1Frag;
        const int o = (q >> 3) & 3;
        outh[idx] = (_Float16)(o < dout ? w2[rperm(q >> 6, (q >> 5) & 1, q & 7) * dout + o] : 0.f);
    } else if (idx < kPackedHalves + kBiasFloats) {
        const int q = idx - kPackedHalves;
        outb[q] = q < 128 ? b1[q] : (q - 128 < dout ? b2[q - 128] : 0.f);
    }
}

// Slot payload: density and 12 colour channels of the voxel's merged index.
template <typename PT>
__global__ void k_render_payload(const int32_t* __restrict__ slot_idx, int64_t nslots,
                                 const float* __restrict__ den, const float* __restrict__ col,
                                 int64_t nidx, PT* __restrict__ pay) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s > nslots) return;
    int64_t id = s < nslots ? slot_idx[s] : 0;  // slot nslots: index 0 (missing leaves)
    if (id < 0 || id >= nidx) id = 0;           // the host checks the range
    PT* p = pay + s * 16;
    p[0] = (PT)den[id];
#pragma unroll
    for (int c = 0; c < 12; ++c) p[1 + c] = (PT)col[id * 12 + c];
    p[13] = p[14] = p[15] = (PT)0.f;
}

// Density cells: for every leaf, the 9 x 9 x 9 trilinear cells that a sample
// whose rounded voxel lies in the leaf can fall in (lower corners -1 .. 7 from
// the leaf's origin on each axis), each with its eight corner densities in the
// corner order of the marches, contiguous.  A march step then needs one
// 16-byte (fp16; two for fp32) load at an address that follows from the leaf
// alone, instead of eight loads behind up to eight more leaf lookups for a
// cell on a leaf's face.  23 MB for 1985 leaves in fp16.
constexpr int kCellSide = 9, kLeafCells = kCellSide * kCellSide * kCellSide;

template <typename PT>
__global__ void k_render_cells(TopoView t, const PT* __restrict__ pay, int64_t nslots,
                               PT* __restrict__ cells) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= t.nleaf * kLeafCells) return;
    const int64_t leaf = c / kLeafCells;
    const int r = (int)(c - leaf * kLeafCells);
    const int i0 = t.origins[3 * leaf] + r / (kCellSide * kCellSide) - 1;
    const int j0 = t.origins[3 * leaf + 1] + (r / kCellSide) % kCellSide - 1;
    const int k0 = t.origins[3 * leaf + 2] + r % kCellSide - 1;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int64_t s = slot_of(t, i0 + ((kCx >> q) & 1), j0 + ((kCy >> q) & 1),
                                  k0 + ((kCz >> q) & 1));
        cells[8 * c + q] = pay[16 * (s < 0 ? nslots : s)];
    }
}

// Workspace of one frame (pvdb_render_workspace_bytes), 256-byte aligned parts.
struct FrameBuffers {
    unsigned long long* total;       // [1] records reserved (may exceed the capacity)
    int32_t* pix_start;              // [HW] first record of the pixel (saturated)
    int32_t* pix_count;              // [HW] pass-1 kept count (records reserved)
    float2* tspan;                   // [HW] pass 2's t range (rewritten t_min, t_max)
    int32_t* pix_written;            // [HW] records pass 2 filled (<= count)
    float* t_last;                   // [HW] transmittance after pass 2
    uint4* pe;                       // [HW][4] PE row: 0 x4, 27 halves, 1
    uint4* rec;                      // [capacity][2] records
    float4* contrib;                 // [capacity] w * sigmoid(raw), per channel
    int64_t capacity;
};

struct RenderArgs {
    TopoView topo;
    const void* payload;
    const void* cells;  // [nleaf][kLeafCells][8] corner densities of the leaves' cells
    int64_t nslots;
    const uint4* packed;
    float* out;
    unsigned long long* counters;  // [3]: pass-1 density gathers, written samples, records
                                   // reserved (may be null)
    FrameBuffers fb;
    float c2w[12];
    float fx, cx, fy, cy;
    float mn[3], ext[3], ws[3], inv_ws[3];
    int32_t H, W, inverse_y;
    int32_t ntx, ntiles;  // the marches' pixel tiles (a wave each): per row, in all
    float near_, stepdist, act_shift, interval, thres, bg, t_stop;
};

// Two floats -> two fp16 (round to nearest even) in one dword, a in the low
// half: one v_cvt_pk_f16_f32.
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    typedef float f2_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2_t){a, b}, half2_t));
}
// relu of two floats as packed fp16: converted first, then one v_pk_max_f16
// (rounding to nearest is monotonic and keeps 0, so this equals converting
// the relu'd values, up to the sign of a zero)
__device__ __forceinline__ uint32_t relu_pack2(float a, float b) {
    const half2_t z = {(_Float16)0.f, (_Float16)0.f};
    const half2_t h = __builtin_bit_cast(half2_t, pack2(a, b));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(h, z));
}

__device__ __forceinline__ float h2f(uint16_t h) {
    return (float)__builtin_bit_cast(_Float16, h);
}

// The eight corner densities of a cell, as loaded (8 fp16 or 8 fp32).
template <bool F32PAY>
struct CellRow {
    uint4 v[F32PAY ? 2 : 1];
    __device__ __forceinline__ void load(const void* cells, uint32_t cell) {
        constexpr int n = F32PAY ? 2 : 1;
        const uint4* p = reinterpret_cast<const uint4*>(cells) + (uint64_t)n * cell;
#pragma unroll
        for (int k = 0; k < n; ++k) v[k] = p[k];
    }
    __device__ __forceinline__ float operator[](int q) const {  // q a constant after unrolling
        if constexpr (F32PAY) {
            const uint4& a = v[q >> 2];
            const uint32_t w[4] = {a.x, a.y, a.z, a.w};
            return __uint_as_float(w[q & 3]);
        } else {
            const uint32_t w[4] = {v[0].x, v[0].y, v[0].z, v[0].w};
            return h2f((uint16_t)(w[q >> 1] >> (16 * (q & 1))));
        }
    }
};

__device__ __forceinline__ f16x8 as_h8(const uint4& v) { return __builtin_bit_cast(f16x8, v); }
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mfma32x32x16h(const uint4& a, const uint4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(as_h8(a), as_h8(b), c, 0, 0, 0);
}
// v_mfma_f32_4x4x4_16b_f16: sixteen 4 x 4 products, block lane / 4; a lane holds
// A[lane % 4][0..3] and B[0..3][lane % 4] of its block and gets D[0..3][lane % 4].
__device__ __forceinline__ f32x4 mfma4x4x4h(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1,
                                            const f32x4& c) {
    typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4, make_uint2(a0, a1)),
                                              __builtin_bit_cast(f16x4, make_uint2(b0, b1)), c, 0, 0, 0);
}

// Leaf index of (i,j,k) through a one-entry cache of its 8^3 block.
struct BlockCache {
    int a = INT32_MIN, b = 0, c = 0;
    int32_t leaf = -1;
    __device__ __forceinline__ int32_t get(const TopoView& t, int i, int j, int k) {
        const int x = i >> 3, y = j >> 3, z = k >> 3;
        if (x != a || y != b || z != c) {
            a = x;
            b = y;
            c = z;
            leaf = leaf_of(t, i, j, k);
        }
        return leaf;
    }
};

// A pixel's ray in the renderer's normalised box coordinates (get_rays,
// renderer.cu:122-167; get_tminmax :50-64).
struct PixelRay {
    float o[3], d[3], step, tmin, tmax;
    float inv_d[3];  // 1 / d (INFINITY for d = 0), for the empty-space exits only
};

__device__ __forceinline__ void pixel_dir(const RenderArgs& A, int px, int py, float* rd) {
    const float pi = (float)px + 0.5f, pj = (float)py + 0.5f;
    const float dx = (pi - A.cx) / A.fx;
    const float dy0 = (pj - A.cy) / A.fy;
    const float dy = A.inverse_y ? dy0 : -dy0;
    const float dz = A.inverse_y ? 1.f : -1.f;
#pragma unroll
    for (int a = 0; a < 3; ++a)
        rd[a] = dx * A.c2w[4 * a] + dy * A.c2w[4 * a + 1] + dz * A.c2w[4 * a + 2];
}

// The pixel's PE row (four zeros, then 27 components of the view direction,
// dvgo.py:91-109 order, and the bias input 1) as fp16, by the pixel's L lanes: each
// takes the sines and cosines of every L-th (axis, frequency) pair.  With one lane a
// pixel evaluating all 24, the wave's other lanes idle, it was a part of the fill
// march: 800 x 800 in fp16 1656 -> 1634 us a frame.
template <int L>
__device__ __forceinline__ void store_pe(const RenderArgs& A, int px, int py, int sub, uint4* row) {
    float rd[3];
    pixel_dir(A, px, py, rd);
    const float len = sqrtf(rd[0] * rd[0] + rd[1] * rd[1] + rd[2] * rd[2]);
    const float inv = 1.f / len;
    const float vd[3] = {rd[0] * inv, rd[1] * inv, rd[2] * inv};
    _Float16* const h = reinterpret_cast<_Float16*>(row) + 4;
    if (sub == 0) {
        reinterpret_cast<uint2*>(row)[0] = make_uint2(0u, 0u);
        h[0] = (_Float16)vd[0];
        h[1] = (_Float16)vd[1];
        h[2] = (_Float16)vd[2];
        h[27] = (_Float16)1.f;  // the bias input
    }
#pragma unroll
    for (int e0 = 0; e0 < 12; e0 += L) {
        const int e = e0 + sub, axis = e >> 2;
        if (e < 12) {
            const float x = (axis == 0 ? vd[0] : axis == 1 ? vd[1] : vd[2]) * (float)(1 << (e & 3));
            h[3 + e] = (_Float16)sinf(x);
            h[15 + e] = (_Float16)cosf(x);
        }
    }
}

__device__ __forceinline__ PixelRay pixel_ray(const RenderArgs& A, int px, int py) {
    PixelRay R;
    float rd[3];
    pixel_dir(A, px, py, rd);
#pragma unroll
    for (int a = 0; a < 3; ++a) R.o[a] = (A.c2w[4 * a + 3] - A.mn[a]) / A.ext[a];
    const float len = sqrtf(rd[0] * rd[0] + rd[1] * rd[1] + rd[2] * rd[2]);
    R.step = A.stepdist / len;
    float lo = -INFINITY, hi = INFINITY;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        R.d[a] = rd[a] / A.ext[a];
        R.inv_d[a] = 1.f / R.d[a];
        const float v = R.d[a] == 0.f ? 1e-6f : R.d[a];
        const float ta = (1.f - R.o[a]) / v, tb = (-R.o[a]) / v;
        lo = a == 0 ? fminf(ta, tb) : fmaxf(lo, fminf(ta, tb));
        hi = a == 0 ? fmaxf(ta, tb) : fminf(hi, fmaxf(ta, tb));
    }
    R.tmin = fmaxf(fminf(lo, 1e9f), A.near_);  // far is forced to 1e9 (plenvdb.h:1008)
    R.tmax = fmaxf(fminf(hi, 1e9f), A.near_);
    return R;
}

// Takes steps t <- t + s (float, round to nearest) while the next t stays
// below tsafe, t < tend and iter < max_iter -- the loop
//     while (t + s < tsafe && t < tend && iter < max_iter) { t += s; ++iter; }
// with the same result, but runs of steps inside one binade [2^(e-1), 2^e)
// of t are taken in O(1): there t is an integer multiple T of the binade's
// ulp u, and t + s rounds to (T + D) u with D = s / u rounded to nearest,
// the same D for every step, unless s / u lies exactly half way between two
// integers (round-half-even would then depend on T's parity) or t + s
// reaches the binade's top.  So k steps give (T + k D) u exactly (an integer
// below 2^24).  k only has to be a lower bound of the loop's count: it is the
// distance to the nearest of the limits over D u in float (at most 2^18 steps
// at a time, where that quotient is off by less than one), less one step; the
// loop takes the rest.
__device__ __forceinline__ void advance_steps(float& t, float s, float tsafe, float tend,
                                              int& iter, int max_iter) {
#pragma unroll 1
    for (int pass = 0; pass < 4; ++pass) {
        if (!(t >= 1e-20f) || !(s > 0.f) || iter >= max_iter) break;
        int e;
        (void)frexpf(t, &e);                   // t in [2^(e-1), 2^e)
        const float q = ldexpf(s, 24 - e);     // s / u, exact
        const float D = rintf(q);
        if (!(q >= 1.f) || !(q < 8388608.f) || fabsf(q - D) == 0.5f) break;
        const float top = ldexpf(1.f, e), lim = fminf(tsafe, tend);
        const float m = (fminf(lim, top) - t) / ldexpf(D, e - 24);
        const int k = (int)fminf(fminf(m, 262144.f) - 1.f, (float)(max_iter - iter));
        if (k < 4) break;
        t = ldexpf((float)((int)ldexpf(t, 24 - e) + k * (int)D), e - 24);
        iter += k;
        if (lim < top) break;
        // at the binade's top: plain steps into the next binade, then again
        for (int z = 0; z < 4 && t + s < tsafe && t < tend && iter < max_iter; ++z) {
            t += s;
            ++iter;
        }
    }
    while (t + s < tsafe && t < tend && iter < max_iter) {
        t += s;
        ++iter;
    }
}

// A march takes its steps L at a time: the L lanes of a ray (consecutive lanes
// of the wave) take its next L steps.  One lane's step: t is the reference's
// running float sum (the steps before it added one by one), `hit` whether the
// sample lies in the box and its rounded voxel is active (isActive(Round(xyz)),
// rintf, half to even, NanoVDB.h:774-779).
template <bool F32PAY>
struct Step {
    float t;
    bool hit;
    int i0, j0, k0;  // the sample's cell (int() truncation, renderer.cu:271-300)
    float u, v, w;
    CellRow<F32PAY> den;
    float te;        // in a missing leaf: t at the exit of the empty cube around it
};

template <bool F32PAY, int L>
__device__ __forceinline__ Step<F32PAY> march_step(const RenderArgs& A, const PixelRay& R,
                                                   float t0, int iter, float tend, int max_iter,
                                                   BlockCache& bc) {
    const int sub = (int)(threadIdx.x & (L - 1));
    Step<F32PAY> s;
    float t = t0, before = t0;
#pragma unroll
    for (int k = 0; k < L; ++k) {
        if (k <= sub) {
            before = t;
            t += R.step;
        }
    }
    s.t = t;
    s.hit = false;
    s.te = -INFINITY;
    const float p0 = R.o[0] + t * R.d[0], p1 = R.o[1] + t * R.d[1], p2 = R.o[2] + t * R.d[2];
    const bool in = p0 >= 0.f && p1 >= 0.f && p2 >= 0.f && p0 <= 1.f && p1 <= 1.f && p2 <= 1.f;
    if (!(in && before < tend && iter + sub < max_iter)) return s;
    const float x = p0 * A.ws[0], y = p1 * A.ws[1], z = p2 * A.ws[2];
    const int vi = (int)rintf(x), vj = (int)rintf(y), vk = (int)rintf(z);
    const int32_t l = bc.get(A.topo, vi, vj, vk);
    if (l < 0) {
        // Empty space: the rounded position is in a missing leaf, and by the
        // empty-run map no leaf lies within r - 1 cells of it, so every step
        // until the ray leaves the rounding box of that cube of cells,
        // [8(L - r + 1) - 0.5, 8(L + r) - 0.5), is rejected by this same test.
        const int c[3] = {vi >> 3, vj >> 3, vk >> 3};
        const int r = empty_run(A.topo, c[0], c[1], c[2]);
        float te = INFINITY;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (R.d[a] == 0.f) continue;
            const float xb = R.d[a] > 0.f ? 8.f * (float)(c[a] + r) - 0.5f
                                          : 8.f * (float)(c[a] - r + 1) - 0.5f;
            te = fminf(te, (xb * A.inv_ws[a] - R.o[a]) * R.inv_d[a]);
        }
        s.te = te;
        return s;
    }
    s.i0 = (int)x;  // x >= 0 here: int() == floor
    s.j0 = (int)y;
    s.k0 = (int)z;
    // the mask word and the cell are loaded together: both follow from the leaf
    // (the host keeps nleaf below 2^22, so the cell's index fits 32 bits)
    const int off = voxel_offset(vi, vj, vk);
    const uint64_t word = A.topo.masks[(int64_t)l * 8 + (off >> 6)];
    s.den.load(A.cells, (uint32_t)l * kLeafCells +
                            (uint32_t)(((s.i0 - (vi & ~7) + 1) * kCellSide +
                                        (s.j0 - (vj & ~7) + 1)) * kCellSide +
                                       (s.k0 - (vk & ~7) + 1)));
    s.hit = (word >> (off & 63)) & 1ull;
    s.u = x - (float)s.i0;
    s.v = y - (float)s.j0;
    s.w = z - (float)s.k0;
    return s;
}

// Lane j's value in each group of L consecutive lanes (j uniform).
template <int L, int J>
__device__ __forceinline__ float group_read(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(
        __builtin_bit_cast(int, x), (J << 5) | (0x1f & ~(L - 1))));
}

// f(0), ..., f(L - 1), the index a compile-time constant.
template <int L, typename F, int K = 0>
__device__ __forceinline__ void for_lanes(F&& f) {
    if constexpr (K < L) {
        f(std::integral_constant<int, K>{});
        for_lanes<L, F, K + 1>(static_cast<F&&>(f));
    }
}

// The next L steps of every ray of the wave: returns the ray's hits as bits and
// moves t past the steps.  Missing leaves are stepped over with the t += step
// accumulation alone (in closed form, advance_steps), stopping two steps short
// of the computed exit, which covers its rounding (the exit is formed with
// reciprocals: a relative error of a few ulps, far inside the two steps); t
// stays the reference's running sum and the set of tested steps is unchanged.
template <bool F32PAY, int L>
__device__ __forceinline__ uint32_t next_steps(const RenderArgs& A, const PixelRay& R, float& t,
                                               int& iter, float tend, int max_iter,
                                               BlockCache& bc, Step<F32PAY>& s) {
    const int g0 = (int)(threadIdx.x & 63 & ~(L - 1));
    s = march_step<F32PAY, L>(A, R, t, iter, tend, max_iter, bc);
    const uint32_t hits = (uint32_t)(__ballot(s.hit) >> g0) & ((1u << L) - 1);
    // the state after these steps; the last one's empty cube is stepped over
    t = group_read<L, L - 1>(s.t);
    iter += L;
    const float te = group_read<L, L - 1>(s.te);
    if (te > t) advance_steps(t, R.step, te - 2.f * R.step, tend, iter, max_iter);
    return hits;
}

__device__ __forceinline__ int march_cap(const PixelRay& R, float t0, float t1) {
    // the reference loop ends when t reaches its bound; the cap only guards
    // steps too small to advance t
    const float span = (t1 - t0) / R.step;
    return (span >= 0.f) ? (int)fminf(span * 1.0625f + 16.f, 16777216.f) : 0;
}

// The pixel of a lane of tile `tile`: a wave's 64 / L pixels, L lanes each, as a
// block of 4 x 4, 4 x 2 or 2 x 2 (row-major tiles).
template <int L>
struct TileShape {
    static_assert(L == 4 || L == 8 || L == 16, "lanes per ray");
    static constexpr int w = L <= 8 ? 4 : 2, h = 64 / L / w;
};
struct TilePixel {
    int px, py;
    bool valid;
    int64_t pix;
};
template <int L>
__device__ __forceinline__ TilePixel tile_pixel(const RenderArgs& A, int tile, int lane) {
    using S = TileShape<L>;
    const int p = lane / L;
    TilePixel P;
    P.px = (tile % A.ntx) * S::w + p % S::w;
    P.py = (tile / A.ntx) * S::h + p / S::w;
    P.valid = P.px < A.W && P.py < A.H;
    P.pix = (int64_t)P.py * A.W + P.px;
    return P;
}

__device__ __forceinline__ void wave_count_add(unsigned long long* dst, unsigned long long v,
                                               int lane) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if (lane == 0 && v) atomicAdd(dst, v);
}

// Both marches are bound by VALU issue at 800 x 800 (318M and 219M wave
// instructions; the search for the next samples is about half of them, powf a
// quarter) and by the waves' chains of dependent loads in small frames.  With a
// lane per pixel, one step at a time and eight corner loads the pair took
// 1970 us at 800 x 800 and 1406 us at 203 x 151 (fp32), now about 950 and 250.
//
// Pass 1, first_look_merged (renderer.cu:222-268): counts the kept samples with
// trigetDensity's summation order and records the rewritten t range: the first
// kept t minus one step, and the t of the early stop (or the box exit).
template <bool F32PAY, int L>
__global__ void __launch_bounds__(kMarchThreads) k_render_count(RenderArgs A) {
    const int lane = threadIdx.x & 63, sub = lane & (L - 1);
    const int tile = blockIdx.x * (kMarchThreads / 64) + (threadIdx.x >> 6);
    if (tile >= A.ntiles) return;  // uniform over the wave
    const FrameBuffers& F = A.fb;
    const TilePixel tp = tile_pixel<L>(A, tile, lane);
    uint32_t n_gather = 0;
    if (tp.valid) {
        const PixelRay R = pixel_ray(A, tp.px, tp.py);
        BlockCache bc;
        float t = R.tmin, T = 1.f, tmin2 = R.tmin, tmax2 = R.tmax;
        int cnt = 0, iter = 0;
        const int cap1 = march_cap(R, R.tmin, R.tmax);
        bool done = false;
        Step<F32PAY> s;
        while (!done && t < R.tmax && iter < cap1) {
            const uint32_t hits = next_steps<F32PAY, L>(A, R, t, iter, R.tmax, cap1, bc, s);
            if (!hits) continue;
            float alpha = 0.f;
            if (s.hit) {
                // trigetDensity order (:191-220): res += den * (1-u) * (1-v) * (1-w), ...
                float sig = 0.f;
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float a = ((kCx >> q) & 1) ? s.u : 1.f - s.u;
                    const float b = ((kCy >> q) & 1) ? s.v : 1.f - s.v;
                    const float e = ((kCz >> q) & 1) ? s.w : 1.f - s.w;
                    sig = sig + ((s.den[q] * a) * b) * e;
                }
                alpha = 1.f - powf(1.f + expf(sig + A.act_shift), -A.interval);
            }
            // the samples of the batch in step order, every lane of the ray alike
            // (selects: the ray's samples rarely agree with its neighbours')
            for_lanes<L>([&](auto k) {
                const float al = group_read<L, k.value>(alpha);
                const float tk = group_read<L, k.value>(s.t);
                const bool on = !done && ((hits >> k.value) & 1u);
                n_gather += on ? 1u : 0u;
                const bool kept_a = on && !(al <= A.thres);
                const float wt = T * al;
                T = kept_a ? T * (1.f - al) : T;
                const bool kept = kept_a && !(wt <= A.thres);
                tmin2 = kept && cnt == 0 ? tk - R.step : tmin2;
                cnt += kept ? 1 : 0;
                const bool stop = kept && T < A.t_stop;
                tmax2 = stop ? tk : tmax2;
                done = done || stop;
            });
        }
        if (sub == 0) {
            F.pix_count[tp.pix] = cnt;
            F.tspan[tp.pix] = make_float2(tmin2, tmax2);
        }
    }
    if (A.counters) wave_count_add(A.counters, sub == 0 ? (unsigned long long)n_gather : 0, lane);
}

// Pass 2, ray_marching_merged (renderer.cu:312-367), from the rewritten t_min
// to t_max with trigetDensity2's summation order: the tile reserves its records
// with one atomic (pass 1's counts scanned across the wave) and writes one
// 32-byte record per kept sample (its cell, fractions, weight and pixel), at
// most pass 1's count of them, contiguous per pixel.
template <bool F32PAY, int L>
__global__ void __launch_bounds__(kMarchThreads) k_render_fill(RenderArgs A) {
    const int lane = threadIdx.x & 63, sub = lane & (L - 1);
    const int tile = blockIdx.x * (kMarchThreads / 64) + (threadIdx.x >> 6);
    if (tile >= A.ntiles) return;  // uniform over the wave
    const FrameBuffers& F = A.fb;
    const TilePixel tp = tile_pixel<L>(A, tile, lane);
    const int cnt = tp.valid ? F.pix_count[tp.pix] : 0;
    int incl = sub == 0 ? cnt : 0;  // a pixel counts once, at its first lane
#pragma unroll
    for (int dd = 1; dd < 64; dd <<= 1) {
        const int o = __shfl_up(incl, dd, 64);
        if (lane >= dd) incl += o;
    }
    const int tile_total = __shfl(incl, 63, 64);
    unsigned long long base = 0;
    if (lane == 0 && tile_total > 0) base = atomicAdd(F.total, (unsigned long long)tile_total);
    base = __shfl(base, 0, 64);
    const int64_t start = (int64_t)base + (incl - cnt);  // the same in all of a pixel's lanes

    int r = 0;
    float T = 1.f;
    if (cnt > 0) {
        const PixelRay R = pixel_ray(A, tp.px, tp.py);
        const float2 span = F.tspan[tp.pix];
        const float tmax2 = span.y;
        BlockCache bc;
        float t = span.x;
        int iter = 0;
        const int cap2 = march_cap(R, span.x, tmax2);
        Step<F32PAY> s;
        while (t < tmax2 && iter < cap2) {
            const uint32_t hits = next_steps<F32PAY, L>(A, R, t, iter, tmax2, cap2, bc, s);
            if (!hits) continue;
            float alpha = 0.f;
            if (s.hit) {
                float sc[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    const float a = ((kCx >> q) & 1) ? s.u : 1.f - s.u;
                    const float b = ((kCy >> q) & 1) ? s.v : 1.f - s.v;
                    const float e = ((kCz >> q) & 1) ? s.w : 1.f - s.w;
                    sc[q] = (a * b) * e;
                }
                // trigetDensity2 order (:271-300): sum of den * scale, left to right
                float sig = s.den[0] * sc[0];
#pragma unroll
                for (int q = 1; q < 8; ++q) sig = sig + s.den[q] * sc[q];
                alpha = 1.f - powf(1.f + expf(sig + A.act_shift), -A.interval);
            }
            int at = -1;  // this lane's record
            float mine = 0.f;
            for_lanes<L>([&](auto k) {
                const float al = group_read<L, k.value>(alpha);
                const bool kept_a = ((hits >> k.value) & 1u) && !(al <= A.thres);
                const float wt = T * al;
                T = kept_a ? T * (1.f - al) : T;
                const bool kept = kept_a && !(wt <= A.thres);
                at = kept && k.value == sub ? r : at;
                mine = kept && k.value == sub ? wt : mine;
                r += kept ? 1 : 0;  // may pass pass 1's count; those are not written
            });
            if (at >= 0 && at < cnt) {
                // the sample's cell and fractions
                const int64_t q = start + at;
                if (q < F.capacity) {
                    F.rec[2 * q] = make_uint4((uint32_t)s.i0, (uint32_t)s.j0, (uint32_t)s.k0,
                                              __float_as_uint(s.u));
                    F.rec[2 * q + 1] = make_uint4(__float_as_uint(s.v), __float_as_uint(s.w),
                                                  __float_as_uint(mine), (uint32_t)tp.pix);
                }
            }
        }
    }
    const int written = r < cnt ? r : cnt;
    // reserved records pass 2 did not fill: no cell (i0 = -1), zero weight
    for (int k = written + sub; k < cnt; k += L) {
        const int64_t q = start + k;
        if (q < F.capacity) {
            F.rec[2 * q] = make_uint4(0xffffffffu, 0u, 0u, 0u);
            F.rec[2 * q + 1] = make_uint4(0u, 0u, 0u, (uint32_t)tp.pix);
        }
    }
    if (tp.valid && sub == 0) {
        F.pix_start[tp.pix] = (int32_t)(start < kMaxRecords ? start : kMaxRecords);
        F.pix_written[tp.pix] = written;
        F.t_last[tp.pix] = cnt > 0 ? T : 1.f;
    }
    if (cnt > 0) store_pe<L>(A, tp.px, tp.py, sub, F.pe + 4 * tp.pix);  // 0 outside the frame
    if (A.counters)
        wave_count_add(A.counters + 1, sub == 0 ? (unsigned long long)written : 0, lane);
}

// The records' colour and the MLP over them: a wavefront takes 32 records
// through the network by itself, activations in registers (the D fragment of
// v_mfma_f32_32x32x16_f16, lane (h, n): features 32T + 8q + 4h + i of sample n, is the
// next layer's B fragment under the K order of rperm).  The colour (trigetColor,
// renderer.cu:303-310) is gathered ahead, four corners to a lane and the other four
// in the lane's other half, under the MFMAs of the group before, so the features
// never see memory.  Each record's contribution is w / (1 + exp(-raw)) per channel
// (final_render, renderer.cu:112-119).  Records: (i0, j0, k0, u | v, w, weight,
// pixel); i0 = -1 marks a reserved record without a sample (no contribution).
//
// What bounds it: the CU's address unit and L1, one row part a lane and cycle (590
// cycles a group, 68% of the time at 800 x 800); the group's 44 MFMAs of 32 cycles
// of its SIMD's matrix core and 440 vector instructions of 4 run beside it (44% and
// 50%).  Three wavefronts per SIMD (fp16 payload) cover most of the loads' latency.
//
// Measured against a gather kernel of a thread per record, which wrote the features
// back into the records, and an MLP kernel with four 16-sample tiles a wavefront:
// 800 x 800, fp16 365 + 572 -> 719 us (the frame 1880 -> 1604 us); 203 x 151, fp32
// 34 + 45 -> 62 us (352 -> 325 us).
template <bool F32PAY>
__global__ void __launch_bounds__(64 * kMlpWaves, F32PAY ? 2 : 3) k_render_mlp(RenderArgs A) {
    constexpr int kRow = F32PAY ? 4 : 2;  // 16-byte parts of a colour row
    __shared__ RenderSmem sm;
    const FrameBuffers& F = A.fb;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = (int)(threadIdx.x & 63), n = lane & 31, h = lane >> 5;
    const unsigned long long tot = *F.total;
    if (A.counters && blockIdx.x == 0 && threadIdx.x == 0) A.counters[2] = tot;
    const int64_t total = (int64_t)(tot < (unsigned long long)F.capacity ? tot : F.capacity);
    if (total <= 0) return;
    const int64_t ngroups = (total + 31) / 32, stride = (int64_t)gridDim.x * kMlpWaves;
    const TopoView& topo = A.topo;

    // the group two ahead: its records (the last record again past the end)
    uint4 ra, rb;
    auto load_records = [&](int64_t grp) {
        const int64_t q = min(min(grp, ngroups - 1) * 32 + n, total - 1);
        ra = F.rec[2 * q];
        rb = F.rec[2 * q + 1];
    };
    // the next group: slots and weights of this lane's four corners (4h .. 4h + 3 of the
    // corner walk: x offset h, the y and z offsets mirrored in y), weight, pixel
    int32_t slot[4];
    float sc[4], nweight;
    uint32_t npix;
    auto lookup = [&]() {
        const int i0 = (int)ra.x, j0 = (int)ra.y, k0 = (int)ra.z;
        const float u = __uint_as_float(ra.w), v = __uint_as_float(rb.x), w = __uint_as_float(rb.y);
        nweight = i0 >= 0 ? __uint_as_float(rb.z) : -1.f;  // no sample's weight is negative
        npix = rb.w;
        const float a = h ? u : 1.f - u;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int dy = (c >> 1) ^ h, dz = (c & 1) ^ (c >> 1);
            sc[c] = (a * (dy ? v : 1.f - v)) * (dz ? w : 1.f - w);
            const int i = i0 + h, j = j0 + dy, k = k0 + dz;
            int32_t leaf;
            if (topo.two_level) {  // uniform over the frame
                leaf = leaf_of(topo, i, j, k);
            } else {  // leaf_of's lookup without a branch
                const int la = (i >> 3) - topo.lo0, lb = (j >> 3) - topo.lo1, lc = (k >> 3) - topo.lo2;
                const bool inside = (unsigned)la < (unsigned)topo.d0 && (unsigned)lb < (unsigned)topo.d1 &&
                                    (unsigned)lc < (unsigned)topo.d2;
                leaf = topo.table[inside ? (la * topo.d1 + lb) * topo.d2 + lc : 0];
                leaf = inside ? leaf : -1;
            }
            slot[c] = leaf < 0 ? (int32_t)A.nslots : leaf * 512 + voxel_offset(i, j, k);
        }
    };
    uint4 raw[2][kRow];  // the colour rows of corners 2 pair, 2 pair + 1
    auto fetch = [&](int pair) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const uint4* src = reinterpret_cast<const uint4*>(A.payload) + (int64_t)slot[2 * pair + c] * kRow;
#pragma unroll
            for (int k = 0; k < kRow; ++k) raw[c][k] = src[k];
        }
    };
    float v[12];  // this lane's corners' weighted colour
    auto weigh = [&](int pair) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const float s = sc[2 * pair + c];
            const uint32_t* r = reinterpret_cast<const uint32_t*>(raw[c]);
#pragma unroll
            for (int ch = 0; ch < 12; ++ch) {
                const int e = ch + 1;  // element 0 is the density
                const float x = F32PAY ? __uint_as_float(r[e]) : h2f((uint16_t)(r[e >> 1] >> (16 * (e & 1))));
                v[ch] = pair == 0 && c == 0 ? x * s : fmaf(x, s, v[ch]);
            }
        }
    };
    uint4 pe2, pe4;  // the pixel's encoding: chunk 2 + h, chunk 4, and chunk 1's half
    uint2 peb;
    auto fetch_pe = [&]() {
        const uint4* row = F.pe + 4 * (int64_t)npix;
        pe2 = row[1 + h];
        pe4 = row[3];
        peb = reinterpret_cast<const uint2*>(row)[1];
    };
    uint4 xb[3];  // a group's X fragments: columns 8h, 16 + 8h, 32 + 8h
    auto form_x = [&]() {
        // the two lane halves' sums: half 0 is left with features 0..7, half 1 with 8..11
        float f[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const auto r = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(v[c]), __float_as_uint(v[c < 4 ? c + 8 : c]), false, false);
            f[c] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
        xb[0] = make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), h ? peb.x : pack2(f[4], f[5]),
                           h ? peb.y : pack2(f[6], f[7]));
        xb[1] = pe2;
        xb[2] = make_uint4(h ? 0u : pe4.x, h ? 0u : pe4.y, h ? 0u : pe4.z, h ? 0u : pe4.w);
    };

    int64_t grp = (int64_t)wv * gridDim.x + blockIdx.x;
    load_records(grp);
    {
        uint4* dst = reinterpret_cast<uint4*>(&sm);
        for (int e = threadIdx.x; e < kPackedBytes / 16; e += 64 * kMlpWaves) dst[e] = A.packed[e];
    }
    lookup();
    load_records(grp + stride);
    fetch(0);
    weigh(0);
    fetch(1);
    fetch_pe();
    weigh(1);
    form_x();
    __syncthreads();  // the weights; from here on the wavefronts run on their own
    const uint4* const w0p = sm.w0 + 128 * h + n;
    const uint4* const w1p = sm.w1 + lane;
    const uint4* const w2p = sm.w2 + 4 * h + (n & 3);
    const float* const b1p = sm.b + 4 * h;
    const float b2a = sm.b[128 + h], b2b = sm.b[130];

    for (; grp < ngroups; grp += stride) {
        const float weight = nweight;
        lookup();
        load_records(grp + 2 * stride);
        uint32_t h0[8][4], h1[4];  // layer 1's B fragments [k-step][dword], layer 2's of one k-step
        f32x16 c, d;               // a tile in the making, the one before
        f32x4 lg = {0.f, 0.f, 0.f, 0.f};
        const f32x16 zero = {};
        auto pair0 = [&](int T, int j) {
            h0[2 * T + (j >> 2)][j & 3] = relu_pack2(d[2 * j], d[2 * j + 1]);
        };
        uint4 w2f;
        auto pair1 = [&](int T, int j) {
            if ((j & 3) == 0) w2f = w2p[8 * (2 * T + (j >> 2))];
            h1[j & 3] = relu_pack2(d[2 * j], d[2 * j + 1]);
            if ((j & 3) == 3) {  // layer 2's k-step 2T + j / 4
                lg = mfma4x4x4h(w2f.x, w2f.y, h1[0], h1[1], lg);
                lg = mfma4x4x4h(w2f.z, w2f.w, h1[2], h1[3], lg);
            }
        };
        // ---- layer 0; the next group's first corners are fetched from here on ----
        uint4 f0[3] = {w0p[0], w0p[256]};  // weight fragments, read two steps ahead
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            if (T == 2) fetch(0);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int s = 3 * T + k;
                if (s < 10) f0[(s + 2) % 3] = w0p[256 * ((s + 2) % 3) + 32 * ((s + 2) / 3)];
                c = mfma32x32x16h(f0[s % 3], xb[k], k == 0 ? zero : c);
                if (T > 0) {
                    pair0(T - 1, 3 * k);
                    pair0(T - 1, 3 * k + 1);
                    if (k < 2) pair0(T - 1, 3 * k + 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            d = c;
        }
        // ---- layer 1; layer 2 over its tiles ----
        uint4 f1[3] = {w1p[0], w1p[64]};
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            if (T == 1) {
                weigh(0);
                fetch(1);
                fetch_pe();
            }
            if (T == 3) weigh(1);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 b = *reinterpret_cast<const float4*>(b1p + 32 * T + 8 * q);
                c[4 * q] = b.x;
                c[4 * q + 1] = b.y;
                c[4 * q + 2] = b.z;
                c[4 * q + 3] = b.w;
            }
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                const int s = 8 * T + ks;
                if (s < 30) f1[(s + 2) % 3] = w1p[64 * (s + 2)];
                c = mfma32x32x16h(f1[s % 3], make_uint4(h0[ks][0], h0[ks][1], h0[ks][2], h0[ks][3]), c);
                if (T > 0) {
                    pair1(T - 1, ks);
                } else if (ks < 4) {  // the last layer-0 tile is k-steps 6 and 7's input
                    pair0(3, 2 * ks);
                    pair0(3, 2 * ks + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            d = c;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) pair1(3, j);
        form_x();
        // the lane halves' logits: half h finishes channel h, half 0 channel 2 too (half 1
        // writes the unused fourth); w * sigmoid(raw) with the hardware exp and reciprocal
        // (a few ulps, far inside the fp16 MLP's own rounding)
        const auto r01 = __builtin_amdgcn_permlane32_swap(__float_as_uint(lg[0]),
                                                          __float_as_uint(lg[1]), false, false);
        const float x = __uint_as_float(r01[0]) + __uint_as_float(r01[1]) + b2a;
        const float y = lg[2] + __shfl_xor(lg[2], 32, 64) + b2b;
        const int64_t q = grp * 32 + n;
        if (q < total) {
            float* dst = reinterpret_cast<float*>(F.contrib + q) + h;
            const bool live = weight != -1.f;
            dst[0] = live ? weight * __builtin_amdgcn_rcpf(1.f + __expf(-x)) : 0.f;
            dst[2] = live && h == 0 ? weight * __builtin_amdgcn_rcpf(1.f + __expf(-y)) : 0.f;
        }
    }
}

// Pixel colour: T_last * bg + the pixel's contributions in sample order.
constexpr int kCompLanes = 8;  // lanes per pixel in k_render_composite

__global__ void __launch_bounds__(256) k_render_composite(RenderArgs A) {
    // lane j of a pixel's eight sums the pixel's records j, j + 8, ... (the
    // eight read 128 contiguous bytes per step), then the eight add up their
    // sums; every lane takes part in the exchange (no early exit)
    const int64_t p = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kCompLanes;
    const int j = (int)(threadIdx.x & (kCompLanes - 1));
    const bool on = p < (int64_t)A.H * A.W;  // uniform over a pixel's lanes
    const FrameBuffers& F = A.fb;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
    if (on) {
        const unsigned long long tot = *F.total;
        const int64_t n = (int64_t)(tot < (unsigned long long)F.capacity ? tot : F.capacity);
        const int64_t s = F.pix_start[p];
        const int wn = F.pix_written[p];
        for (int k = j; k < wn; k += kCompLanes) {
            const int64_t q = s + k;
            if (q >= n) break;
            const float4 c = F.contrib[q];
            a0 = a0 + c.x;
            a1 = a1 + c.y;
            a2 = a2 + c.z;
        }
    }
#pragma unroll
    for (int d = 1; d < kCompLanes; d <<= 1) {
        a0 += __shfl_xor(a0, d, 64);
        a1 += __shfl_xor(a1, d, 64);
        a2 += __shfl_xor(a2, d, 64);
    }
    if (on && j == 0) {
        const float last = F.t_last[p] * A.bg;
        A.out[3 * p] = last + a0;
        A.out[3 * p + 1] = last + a1;
        A.out[3 * p + 2] = last + a2;
    }
}

__global__ void k_render_reset(unsigned long long* total, unsigned long long* counters) {
    if (threadIdx.x == 0) *total = 0ull;
    if (counters && threadIdx.x < 3) counters[threadIdx.x] = 0ull;
}

inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// Optional device timing of the three kernels (HIP events around each launch).
struct RenderTimer {
    bool enabled = false;
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> open;
    double total_ms[3] = {0, 0, 0};
};
RenderTimer g_rtimer;

struct RenderStage {
    int stage;
    hipStream_t s;
    hipEvent_t a = nullptr, b = nullptr;
    RenderStage(int st, hipStream_t str) : stage(st), s(str) {
        if (!g_rtimer.enabled) return;
        hipEventCreate(&a);
        hipEventCreate(&b);
        hipEventRecord(a, s);
    }
    ~RenderStage() {
        if (!g_rtimer.enabled || !a) return;
        hipEventRecord(b, s);
        g_rtimer.open.push_back({stage, {a, b}});
    }
};

// Payload of (nslots + 1) slots: the slot rows (32 or 64 bytes: density and
// 12 colour channels), then the leaves' density cells (16 or 32 bytes a cell).
struct PayloadLayout {
    size_t cells, bytes;
};
PayloadLayout payload_layout(const TopoView& t, int32_t payload_f32) {
    const size_t n = (size_t)t.nleaf * 512 + 1, es = payload_f32 ? 4 : 2;
    PayloadLayout L;
    L.cells = align256(n * 16 * es);
    L.bytes = align256(L.cells + (size_t)t.nleaf * kLeafCells * 8 * es);
    return L;
}

struct FrameLayout {
    size_t total, start, count, tspan, written, tlast, pe, rec, contrib, bytes;
};

FrameLayout frame_layout(int64_t hw, int64_t capacity) {
    FrameLayout L;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o = align256(o + bytes);
        return at;
    };
    L.total = take(8);
    L.start = take(4 * (size_t)hw);
    L.count = take(4 * (size_t)hw);
    L.tspan = take(8 * (size_t)hw);
    L.written = take(4 * (size_t)hw);
    L.tlast = take(4 * (size_t)hw);
    L.pe = take(64 * (size_t)hw);
    L.rec = take(32 * (size_t)capacity);
    L.contrib = take(16 * (size_t)capacity);
    L.bytes = o;
    return L;
}

FrameBuffers frame_buffers(void* ws, int64_t hw, int64_t capacity) {
    const FrameLayout L = frame_layout(hw, capacity);
    uint8_t* b = reinterpret_cast<uint8_t*>(ws);
    FrameBuffers F;
    F.total = reinterpret_cast<unsigned long long*>(b + L.total);
    F.pix_start = reinterpret_cast<int32_t*>(b + L.start);
    F.pix_count = reinterpret_cast<int32_t*>(b + L.count);
    F.tspan = reinterpret_cast<float2*>(b + L.tspan);
    F.pix_written = reinterpret_cast<int32_t*>(b + L.written);
    F.t_last = reinterpret_cast<float*>(b + L.tlast);
    F.pe = reinterpret_cast<uint4*>(b + L.pe);
    F.rec = reinterpret_cast<uint4*>(b + L.rec);
    F.contrib = reinterpret_cast<float4*>(b + L.contrib);
    F.capacity = capacity;
    return F;
}

template <typename PT>
void build_payload(const TopoView& t, const int32_t* slot_idx, const float* den, const float* col,
                   int64_t nidx, uint8_t* p, const PayloadLayout& L, hipStream_t s) {
    const int64_t nslots = t.nleaf * 512;
    PT* pay = reinterpret_cast<PT*>(p);
    hipLaunchKernelGGL(k_render_payload<PT>, dim3(pvdb_blocks(nslots + 1, 256)), dim3(256), 0, s,
                       slot_idx, nslots, den, col, nidx, pay);
    hipLaunchKernelGGL(k_render_cells<PT>, dim3(pvdb_blocks(t.nleaf * kLeafCells, 256)), dim3(256),
                       0, s, t, pay, nslots, reinterpret_cast<PT*>(p + L.cells));
}

}  // namespace

extern "C" {

int64_t pvdb_render_weights_bytes(void) { return kPackedBytes; }

int pvdb_render_pack_weights(const float* w0, const float* b0, const float* w1, const float* b1,
                             const float* w2, const float* b2, int32_t dcol, int32_t dpe,
                             int32_t dhid, int32_t dout, void* packed, void* stream) {
    PVDB_CHECK_ARG(w0 && b0 && w1 && b1 && w2 && b2 && packed, "null pointer");
    PVDB_CHECK_ARG(dcol == 12 && dpe == 27 && dhid == kHid && dout == 3,
                   "unsupported MLP shape: the renderer takes dcol 12, dpe 27, dhid 128, dout 3");
    uint8_t* p = reinterpret_cast<uint8_t*>(packed);
    const int n = kPackedHalves + kBiasFloats;
    hipLaunchKernelGGL(k_render_pack, dim3(pvdb_blocks(n, 256)), dim3(256), 0,
                       (hipStream_t)stream, w0, b0, w1, b1, w2, b2, dcol, dpe, dout,
                       reinterpret_cast<_Float16*>(p),
                       reinterpret_cast<float*>(p + kPackedHalves * 2));
    PVDB_LAUNCHED("k_render_pack");
    return PVDB_OK;
}

int64_t pvdb_render_payload_bytes(const pvdb_topology* topo, int32_t payload_f32) {
    if (!topo) return -1;
    return (int64_t)payload_layout(view_of(topo), payload_f32).bytes;
}

int pvdb_render_build_payload(const pvdb_topology* topo, const int32_t* slot_idx,
                              const float* den, const float* col, int64_t nidx,
                              int32_t payload_f32, void* payload, void* stream) {
    if (!topo) {
        pvdb::set_error("null topology");
        return PVDB_EHANDLE;
    }
    PVDB_CHECK_ARG(slot_idx && den && col && payload, "null pointer");
    PVDB_CHECK_ARG(nidx >= 1, "the data arrays need at least index 0");
    const TopoView tv = view_of(topo);
    const PayloadLayout L = payload_layout(tv, payload_f32);
    uint8_t* p = reinterpret_cast<uint8_t*>(payload);
    hipStream_t st = (hipStream_t)stream;
    if (payload_f32)
        build_payload<float>(tv, slot_idx, den, col, nidx, p, L, st);
    else
        build_payload<_Float16>(tv, slot_idx, den, col, nidx, p, L, st);
    PVDB_LAUNCHED("k_render_payload");
    return PVDB_OK;
}

int64_t pvdb_render_workspace_bytes(int32_t H, int32_t W, int64_t capacity) {
    if (H <= 0 || W <= 0 || capacity < 0 || capacity >= kMaxRecords) return -1;
    return (int64_t)frame_layout((int64_t)H * W, capacity).bytes;
}

int pvdb_render_frame_info(const pvdb_render_desc* d, uint64_t* total, int32_t** pix_count,
                           int32_t** pix_written, int32_t** pix_start) {
    PVDB_CHECK_ARG(d && d->workspace, "null descriptor or workspace");
    const FrameBuffers F = frame_buffers(d->workspace, (int64_t)d->H * d->W, d->capacity);
    if (total) {
        unsigned long long v = 0;
        PVDB_HIP(hipMemcpy(&v, F.total, sizeof(v), hipMemcpyDeviceToHost));
        *total = v;
    }
    if (pix_count) *pix_count = F.pix_count;
    if (pix_written) *pix_written = F.pix_written;
    if (pix_start) *pix_start = F.pix_start;
    return PVDB_OK;
}

}  // extern "C"

namespace {

// The two marches with L lanes per ray: a wave per tile of 64 / L pixels.
template <bool F32PAY, int L>
int launch_marches(RenderArgs A, hipStream_t s) {
    using S = TileShape<L>;
    A.ntx = (A.W + S::w - 1) / S::w;
    A.ntiles = A.ntx * ((A.H + S::h - 1) / S::h);
    const dim3 grid((A.ntiles + kMarchThreads / 64 - 1) / (kMarchThreads / 64));
    hipLaunchKernelGGL((k_render_count<F32PAY, L>), grid, dim3(kMarchThreads), 0, s, A);
    PVDB_LAUNCHED("k_render_count");
    hipLaunchKernelGGL((k_render_fill<F32PAY, L>), grid, dim3(kMarchThreads), 0, s, A);
    PVDB_LAUNCHED("k_render_fill");
    return PVDB_OK;
}

// Lanes per ray by the frame's pixels.  A wave's time is its longest ray's
// chain of dependent steps, so a small frame wants each ray cut into few
// batches (and many waves), while a frame that fills the chip is bound by VALU
// issue and wants few lanes past the rays' ends.  Whole frames, us, at
// 4 / 8 / 16 lanes: 64 x 64 269 / 188 / 151; 203 x 151 344 / 299 / 347;
// 200 x 200 456 / 373 / 386; 400 x 400 702 / 702 / 926; 560 x 560 1053 / 1166 /
// 1699; 800 x 800 1859 / 2304 / - (one and two lanes per ray: 2270 and 1922 at
// 800 x 800, slower below).
template <bool F32PAY>
int launch_marches_sized(const RenderArgs& A, hipStream_t s) {
    const int64_t px = (int64_t)A.H * A.W;
    if (px <= 16384) return launch_marches<F32PAY, 16>(A, s);
    if (px <= 131072) return launch_marches<F32PAY, 8>(A, s);
    return launch_marches<F32PAY, 4>(A, s);
}

// The frame on `ws` (a 256-byte aligned workspace of at least
// pvdb_render_workspace_bytes(H, W, capacity) bytes; the callers check it).
int render_image(const pvdb_topology* topo, const pvdb_render_desc* d, void* ws,
                 hipStream_t stream) {
    for (int a = 0; a < 3; ++a) {
        PVDB_CHECK_ARG(d->reso[a] >= 2, "reso must be at least 2");
        PVDB_CHECK_ARG(d->xyz_max[a] > d->xyz_min[a], "empty bounding box");
    }
    const TopoView t = view_of(topo);
    PVDB_CHECK_ARG(t.nleaf * 512 + 1 < kMaxRecords, "too many leaves for the renderer's slot indices");
    RenderArgs A;
    A.topo = t;
    A.payload = d->payload;
    const PayloadLayout PL = payload_layout(t, d->payload_f32);
    A.cells = reinterpret_cast<const uint8_t*>(d->payload) + PL.cells;
    A.nslots = t.nleaf * 512;
    A.packed = reinterpret_cast<const uint4*>(d->weights);
    A.out = d->out;
    A.counters = reinterpret_cast<unsigned long long*>(d->counters);
    A.fb = frame_buffers(ws, (int64_t)d->H * d->W, d->capacity);
    for (int r = 0; r < 3; ++r)
        for (int c = 0; c < 4; ++c) A.c2w[4 * r + c] = d->c2w[4 * r + c];
    A.fx = d->K[0];
    A.cx = d->K[2];
    A.fy = d->K[4];
    A.cy = d->K[5];
    for (int a = 0; a < 3; ++a) {
        A.mn[a] = d->xyz_min[a];
        A.ext[a] = d->xyz_max[a] - d->xyz_min[a];
        A.ws[a] = (float)(d->reso[a] - 1);
        A.inv_ws[a] = 1.f / A.ws[a];
    }
    A.H = d->H;
    A.W = d->W;
    A.inverse_y = d->inverse_y;
    A.near_ = d->near_;
    A.stepdist = d->stepdist;
    A.act_shift = d->act_shift;
    A.interval = d->interval;
    A.thres = d->fast_color_thres;
    A.bg = d->bg;
    A.t_stop = d->t_stop;
    hipStream_t s = stream;
    hipLaunchKernelGGL(k_render_reset, dim3(1), dim3(64), 0, s, A.fb.total, A.counters);
    PVDB_LAUNCHED("k_render_reset");
    static int ncu = 0;
    if (ncu == 0) {
        int dev = 0;
        PVDB_HIP(hipGetDevice(&dev));
        PVDB_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    }
    {
        RenderStage st(0, s);
        const int rc = d->payload_f32 ? launch_marches_sized<true>(A, s)
                                      : launch_marches_sized<false>(A, s);
        if (rc != PVDB_OK) return rc;
    }
    {
        RenderStage st(1, s);
        // two workgroups a CU, by registers; three for an fp16 payload
        hipLaunchKernelGGL(d->payload_f32 ? k_render_mlp<true> : k_render_mlp<false>, dim3((d->payload_f32 ? 2 : 3) * ncu),
                           dim3(64 * kMlpWaves), 0, s, A);
        PVDB_LAUNCHED("k_render_mlp");
    }
    {
        RenderStage st(2, s);
        hipLaunchKernelGGL(k_render_composite,
                           dim3(pvdb_blocks((int64_t)A.H * A.W * kCompLanes, 256)), dim3(256), 0,
                           s, A);
        PVDB_LAUNCHED("k_render_composite");
    }
    return PVDB_OK;
}

}  // namespace

// Frame workspace of the no-allocation entry point.  The array's name is only
// a host-side handle: host code uses the device address hipGetSymbolAddress
// gives for it, kept per device (each device holds its own copy).
constexpr int64_t kScratchBytes = int64_t(64) << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace {

// Checks shared by both entry points (everything but the workspace).
int check_frame(const pvdb_topology* topo, const pvdb_render_desc* d) {
    if (!topo) {
        pvdb::set_error("null topology");
        return PVDB_EHANDLE;
    }
    PVDB_CHECK_ARG(d && d->payload && d->weights && d->out, "null pointer");
    PVDB_CHECK_ARG(d->H > 0 && d->W > 0 && (int64_t)d->H * d->W < (int64_t(1) << 31),
                   "bad image size");
    PVDB_CHECK_ARG(d->stepdist > 0.f && std::isfinite(d->stepdist), "stepdist must be positive");
    PVDB_CHECK_ARG(d->capacity >= 0 && d->capacity < kMaxRecords,
                   "record capacity must be in [0, 2^31 - 2]");
    return PVDB_OK;
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

int scratch_of_current_device(void** out) {
    int dev = 0;
    PVDB_HIP(hipGetDevice(&dev));
    PVDB_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device ordinal beyond the scratch table");
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        PVDB_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        PVDB_CHECK_ARG(p && reinterpret_cast<uintptr_t>(p) % 256 == 0,
                       "scratch address not 256-byte aligned");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return PVDB_OK;
}

}  // namespace

extern "C" {

int pvdb_render_image(const pvdb_topology* topo, const pvdb_render_desc* d, void* stream) {
    const int rc = check_frame(topo, d);
    if (rc != PVDB_OK) return rc;
    PVDB_CHECK_ARG(d->workspace, "null workspace");
    PVDB_CHECK_ARG(reinterpret_cast<uintptr_t>(d->workspace) % 256 == 0,
                   "workspace must be 256-byte aligned");
    PVDB_CHECK_ARG(d->workspace_bytes >= pvdb_render_workspace_bytes(d->H, d->W, d->capacity),
                   "workspace too small");
    return render_image(topo, d, d->workspace, (hipStream_t)stream);
}

int64_t pvdb_render_noalloc_scratch_bytes(void) { return kScratchBytes; }

int pvdb_render_image_noalloc(const pvdb_topology* topo, const pvdb_render_desc* d,
                              void* stream) {
    const int rc = check_frame(topo, d);
    if (rc != PVDB_OK) return rc;
    const int64_t need = pvdb_render_workspace_bytes(d->H, d->W, d->capacity);
    PVDB_CHECK_ARG(need > 0 && need <= kScratchBytes,
                   "frame does not fit the 64 MiB scratch of pvdb_render_image_noalloc "
                   "(pvdb_render_workspace_bytes(H, W, capacity) must be at most "
                   "pvdb_render_noalloc_scratch_bytes())");
    void* ws = nullptr;
    const int rs = scratch_of_current_device(&ws);
    if (rs != PVDB_OK) return rs;
    return render_image(topo, d, ws, (hipStream_t)stream);
}

int pvdb_render_timing(int32_t enable, double* total_ms3) {
    for (auto& e : g_rtimer.open) {
        hipEventSynchronize(e.second.second);
        float ms = 0.f;
        hipEventElapsedTime(&ms, e.second.first, e.second.second);
        g_rtimer.total_ms[e.first] += ms;
        hipEventDestroy(e.second.first);
        hipEventDestroy(e.second.second);
    }
    g_rtimer.open.clear();
    for (int i = 0; i < 3; ++i) {
        if (total_ms3) total_ms3[i] = g_rtimer.total_ms[i];
        if (enable >= 0) g_rtimer.total_ms[i] = 0;
    }
    if (enable >= 0) g_rtimer.enabled = enable != 0;
    return PVDB_OK;
}

}  // extern "C"
