// Fused step, sample side: the view-dependent RGB MLP (39-128-128-3, ReLU,
// sigmoid; plenvdb/lib/dvgo.py:91-109,354-362) on MFMA, forward and backward,
// over groups of 32 consecutive records.
//
// Activations are computed transposed (features x samples, the samples being an
// MFMA's N dimension):
//   H0^T = relu(W0^T X^T + b0),  H1^T = relu(W1^T H0^T + b1),  L^T = W2^T H1^T + b2
// Weights are held in bf16; gradients and the last
// hidden layer travel as (hi, lo) bf16 pairs, so each product with a weight is
// two MFMAs, which keeps about 16 significant bits where plain bf16 keeps 8
// (plain bf16 inputs put the colour-feature gradients several percent off an
// FP64 evaluation).  The forward's first two products take (hi, mid, lo)
// triples (three MFMAs, fp32's 24 bits): their pre-activations decide the ReLU
// masks the backward applies, and a mask bit that rounds the other way moves a
// sample's feature gradient by a whole term.  dW products (activation x
// gradient) take the hi parts only.
//
// The order of every sum but dW's, which run over samples, is part of the results: the
// bias, then for every 32 inputs the products with their hi, mid and lo parts, eight
// inputs at a time (an MFMA's sum over K is eight terms at a time into the accumulator,
// each eight in no order, so two 32x32x16 are one 16x16x32, bit for bit).  In another
// order about two pre-activations of 190k records end on the other side of zero,
// and colour moments move by up to 1.4e-3 of the largest.  tests/test_gpu_mlp_order.py
// holds the order.
//
// k_mlp_fwd gathers the colour features and writes each record's rgb, ReLU masks
// and bf16 input row (so the backward reads 80 bytes per record instead of
// redoing 8 gathers).  k_mlp_bwd takes each sample's dL/dlogit and dL/dsigma from
// the composite pass, runs g_H1^T = W2 g_L^T, g_H0^T = W1 g_H1^T (masked by
// the forward's ReLU masks), g_X^T = W0[0:12] g_H0^T, recomputes H0 and H1 for the
// dW operands, accumulates dW in registers (one partial per workgroup), and
// writes each record's feature and sigma gradients; the scatter
// (fused_scatter.hip) then adds them to the grids with the "leaf must exist"
// rule (densityvdb.cu:16-27, colorvdb.cu:28-37).  Both kernels load a group's
// records into registers while an earlier group computes.

#include <cstddef>
#include <type_traits>

#include "fused_common.h"
#include "gather.h"
#include "plenvdb_hip.h"

namespace pvdb {
TopoView view_of(const pvdb_topology* t);
}

using namespace pvdb;

namespace {

constexpr int GS = 32;  // records per group

__device__ __forceinline__ bf16x8 as_bf8(const uint4& v) { return __builtin_bit_cast(bf16x8, v); }

// ---- forward -----------------------------------------------------------------
// A wavefront takes a group of 32 records through the whole network by itself:
// its activations never leave its registers, so there is no barrier and no
// exchange between wavefronts once the weights are in LDS.  The D fragment of
// v_mfma_f32_32x32x16_bf16 (lane (h, n), h = lane / 32: rows 8q + 4h + i of
// sample n, q, i < 4) is the next layer's B fragment, K in its natural order, when
// the features stand in layer 0's row order (mlp_feature).  A weight fragment read
// from LDS (8 LDS cycles) covers the three parts of the split activations: 96 cycles
// of its SIMD's matrix core.  X and H0 enter their products as (hi, mid, lo) triples,
// so the pre-activations, and with them the ReLU masks the backward applies,
// carry fp32 precision; H1 enters the logits as (hi, lo) pairs.
//
// X has 40 columns (12 features, 27 encoding inputs, the bias input) in three
// parts.  Stacked along K, behind the ones that meet b0's own split, they are 16 chunks
// of 8 columns, two to a k-step, in the order
//   ones, hi 0 | hi 1, 2 | hi 3, mid 0 | mid 1, 2 | mid 3, lo 0 | lo 1, 2 | lo 3, hi 4 |
//   mid 4, lo 4
// and sit in a tile of the wavefront's own in LDS.
//
// The last group's rows past the records are stored like the others (the
// workspace holds whole groups) and never read.
//
// A lane gathers four corners of its sample's colour, the other lane half the
// other four.  The next group's leaf lookups are issued ahead of layer 0 and
// its colour rows and encoding chunks from there to layer 1's end, so their
// latency runs under the MFMAs; missing leaves and dead samples read rows of
// zeros, which keeps the loop free of branches that the loads would wait in.
//
// What bounds it: a group is 132 MFMAs of 32 cycles of its SIMD's matrix core
// (and 16 of 16) and about 1150 vector instructions of 4 cycles; two wavefronts
// per SIMD (256 registers) overlap them in part.  32x32x16 MFMAs are half as many
// to issue as 16x16x32 ones.  The splits stay an unpacking and a subtraction:
// a dot-product instruction does both at once, but runs on the matrix core
// and does not overlap with MFMAs.  The logits, 3 of 16 rows, use 16x16x32 MFMAs, in
// layer 1's row order two lane swaps from its D fragments.
//
// Measured against four wavefronts that shared a group (32 hidden features each,
// activations exchanged through LDS, three barriers a group): 7.80M records with
// bf16 colour 2029 -> 958 us, 190k with fp32 colour 61.4 -> 37.5 us; 24k, one
// group to a wavefront, 13.8 -> 15.1 us.  On 16x16x32 MFMAs 1204 us.  With the
// gather in the march (features through memory) 900 us, and the march 485 us
// instead of 224.
constexpr int kFwdWaves = 4;
constexpr int kXChunks = 15;
struct alignas(16) SmemFwd {
    uint4 w0[6 * 128];             // [chunk][tile row]: W0^T columns 8c .. 8c + 7; b0's split
    uint4 w1[4 * 9 * 64];          // [row tile][step][lane]: b1's split, then W1^T's A
                                   // fragments of the eight k-steps
    uint4 w2[4 * 4 * 4];           // W2^T rows [tile][group of eight features][logit, zeros]
    uint4 ones;                    // the inputs that the biases' splits are multiplied with
    uint4 x[kFwdWaves][GS][kXChunks];
};

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + expf(-x)); }

// v_mfma_f32_4x4x4_16b_bf16: sixteen 4 x 4 products, block lane / 4.  A lane
// holds A[lane % 4][0..3] and B[0..3][lane % 4] of its block and gets
// D[0..3][lane % 4]: for four logits' weights in A and its own sample's four
// features in B, the lane's own logits.
__device__ __forceinline__ f32x4 mfma4x4x4(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1,
                                           const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4, make_uint2(a0, a1)),
                                                  __builtin_bit_cast(s16x4, make_uint2(b0, b1)), c,
                                                  0, 0, 0);
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ f32x16 mfma32x32x16(const uint4& a, const uint4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf8(a), as_bf8(b), c, 0, 0, 0);
}

// Pins the values' computation to this point: left alone, the compiler defers
// it and keeps the activations that it comes from alive.
__device__ __forceinline__ void pin(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

__device__ __forceinline__ uint4 frag(const uint32_t (&d)[4]) {
    return make_uint4(d[0], d[1], d[2], d[3]);
}

// Orders a wavefront's LDS writes before its own later reads.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// relu as an integer max: a float is > 0 exactly when its bits are > 0 as an
// int, and the max keeps +NaN as torch's relu does (a float max would first
// canonicalize the MFMA output).
__device__ __forceinline__ float relu(float x) {
    return __uint_as_float((uint32_t)max((int32_t)__float_as_uint(x), 0));
}

// The ReLU mask bits of a packed pair of relu'd bf16 values (their hi parts):
// set where the value is not zero, pair p's at bits p and 16 + p.
__device__ __forceinline__ void mask_pair(uint32_t hi, int p, uint32_t& word) {
    uint32_t on;  // as packed integers: the generic form of this min is lowered lane by lane
    asm("v_pk_min_u16 %0, %1, %2" : "=v"(on) : "v"(hi), "s"(0x00010001u));
    word |= on << p;
}

// The network's weights into LDS, by the whole workgroup.
__device__ __forceinline__ void stage_fwd_weights(SmemFwd& sm, const MlpPacked& W) {
    static_assert(offsetof(SmemFwd, w1) == 2 * kImgW1 && offsetof(SmemFwd, w2) == 2 * kImgW2 &&
                      offsetof(SmemFwd, ones) == 2 * kImgOnes && offsetof(SmemFwd, x) == 2 * kFwdImage,
                  "the image is the struct's head");
    uint4* dst = reinterpret_cast<uint4*>(&sm);
#pragma unroll
    for (int k = 0; k < (kFwdImage / 8 + 64 * kFwdWaves - 1) / (64 * kFwdWaves); ++k) {
        const int e = 64 * kFwdWaves * k + (int)threadIdx.x;
        if (e < kFwdImage / 8) dst[e] = W.fwd[e];
    }
}

template <bool BF16COL>
__global__ void __launch_bounds__(64 * kFwdWaves, 2)
    k_mlp_fwd(StepParams P, TopoView topo, const void* color, MlpPacked W, RayBuffers R,
              Records rec) {
    using Raw = std::conditional_t<BF16COL, uint2, float4>;  // one third of a colour row
    __shared__ SmemFwd sm;
    // the wavefront's index as a scalar: record addresses are then scalar bases
    // with lane offsets
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = lane_id(), n = lane & 31, h = lane >> 5;
    const int64_t total = min((int64_t)R.total[0], P.capacity);
    if (total <= 0) return;
    const int64_t ngroups = (total + GS - 1) / GS;
    const int64_t stride = (int64_t)gridDim.x * kFwdWaves;
    uint4* const xr = sm.x[wv][n];  // this lane's sample
    const uint4* const xfirst = h ? &xr[0] : &sm.ones;
    // W0 fragments: this lane's rows of the k-steps' chunk pairs (bias, 0), (1, 2),
    // (3, 0), (3, 4) and (4, 4)
    const uint4* const w0b0 = sm.w0 + (h ? 0 : 128 * 5) + n;
    const uint4* const w012 = sm.w0 + 128 * (1 + h) + n;
    const uint4* const w030 = sm.w0 + (h ? 0 : 128 * 3) + n;
    const uint4* const w034 = sm.w0 + 128 * (3 + h) + n;
    const uint4* const w044 = sm.w0 + 128 * 4 + n;
    const uint4* const w1p = sm.w1 + lane;
    const uint4* const w2p = sm.w2 + 4 * (lane >> 4) + min(lane & 15, 3);

    const int32_t* const none = reinterpret_cast<const int32_t*>(R.zero + 12);  // a leaf index of -1
    // the group two ahead: its records (position, flags); zero flags past the end
    float rx, ry, rz;
    uint32_t rbits;
    auto load_records = [&](int64_t grp) {
        const int64_t q0 = min(grp, ngroups - 1) * GS;
        const float4 p = (rec.xyze + q0)[n];
        rx = p.x;
        ry = p.y;
        rz = p.z;
        const uint32_t b = __float_as_uint((rec.ab + q0)[n].y);
        rbits = n < total - q0 ? b : 0u;
    };
    // the next group: the leaves (-1: none), voxel offsets and weights of this
    // lane's four corners (4h .. 4h + 3 of the corner walk: x offset h, the y
    // and z offsets mirrored in y), and the flags
    int32_t leaf[4];
    uint32_t off[2];  // two to a word
    float sc[4];
    uint32_t nbits;
    auto lookup = [&]() {
        nbits = rbits;
        const bool alive = (rbits & kAliveW) != 0u;
        const Cell cell = make_cell(rx, ry, rz);
        const float a = h ? cell.u : 1.f - cell.u;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int dy = (c >> 1) ^ h, dz = (c & 1) ^ (c >> 1);
            const float b = dy ? cell.v : 1.f - cell.v;
            sc[c] = (a * b) * (dz ? cell.w : 1.f - cell.w);
            const int i = cell.i0 + h, j = cell.j0 + dy, k = cell.k0 + dz;
            const uint32_t vo = (uint32_t)voxel_offset(i, j, k);
            off[c >> 1] = (c & 1) ? off[c >> 1] | (vo << 16) : vo;
            if (topo.two_level) {  // uniform over the grid
                leaf[c] = alive ? leaf_of(topo, i, j, k) : -1;
            } else {  // leaf_of's lookup with a selected address instead of a branch
                const int la = (i >> 3) - topo.lo0, lb = (j >> 3) - topo.lo1, lc = (k >> 3) - topo.lo2;
                const bool inside = alive && (unsigned)la < (unsigned)topo.d0 &&
                                    (unsigned)lb < (unsigned)topo.d1 && (unsigned)lc < (unsigned)topo.d2;
                const int32_t* e = topo.table + ((la * topo.d1 + lb) * topo.d2 + lc);
                leaf[c] = *(inside ? e : none);
            }
        }
    };
    // colour rows of corners 2 pair, 2 pair + 1 (a missing leaf reads the row of zeros)
    Raw raw[2][3];
    auto fetch = [&](int pair, Raw (&raw)[2][3]) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int32_t lf = leaf[2 * pair + c];
            const Raw* src =
                lf >= 0 ? reinterpret_cast<const Raw*>(color) +
                              3 * ((int64_t)lf * 512 + ((off[pair] >> (16 * c)) & 0xffffu))
                        : reinterpret_cast<const Raw*>(R.zero);
            raw[c][0] = src[0];
            raw[c][1] = src[1];
            raw[c][2] = src[2];
        }
    };
    // w[c] = the pair's weighted colour
    auto weigh = [&](int pair, const Raw (&raw)[2][3], float (&w)[12]) {
        const float s0 = sc[2 * pair], s1 = sc[2 * pair + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            float4 c0, c1;
            if constexpr (BF16COL) {
                c0 = make_float4(bf_lo(raw[0][k].x), bf_hi(raw[0][k].x), bf_lo(raw[0][k].y),
                                 bf_hi(raw[0][k].y));
                c1 = make_float4(bf_lo(raw[1][k].x), bf_hi(raw[1][k].x), bf_lo(raw[1][k].y),
                                 bf_hi(raw[1][k].y));
            } else {
                c0 = raw[0][k];
                c1 = raw[1][k];
            }
            w[4 * k + 0] = c0.x * s0 + c1.x * s1;
            w[4 * k + 1] = c0.y * s0 + c1.y * s1;
            w[4 * k + 2] = c0.z * s0 + c1.z * s1;
            w[4 * k + 3] = c0.w * s0 + c1.w * s1;
        }
    };
    // the encoding chunks of the sample's ray (zeros unless it is weight-kept): this
    // lane's halves of k-steps 3..7, and chunk B's columns
    u32x4 pe[5];
    uint2 peb[2];
    auto fetch_pe = [&]() {
        const u32x4* row = reinterpret_cast<const u32x4*>(
            nbits & kAliveW ? R.pe + 96 * (int64_t)(nbits & kRayMask)
                            : reinterpret_cast<const uint16_t*>(R.zero));
        pe[0] = row[1 + h];
        pe[1] = row[5 + h];
        pe[2] = row[9 + h];
        pe[3] = row[3 + 4 * h];
        pe[4] = row[11];
        peb[0] = reinterpret_cast<const uint2*>(row + 4 * h)[1];
        peb[1] = reinterpret_cast<const uint2*>(row + 8 - 4 * h)[1];
    };
    // the sample's X into the wavefront's tile: v holds this lane's four corners
    auto store_x = [&](float (&v)[12]) {
        // the two lane halves' sums: a swap exchanges half of one value's lanes
        // for half of another's, which leaves half h with features 6h .. 6h + 5
        uint32_t hi[3], mi[3], lo[3];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const auto r = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(v[c]), __float_as_uint(v[c + 6]), false, false);
            v[c] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) split3(v[2 * p], v[2 * p + 1], hi[p], mi[p], lo[p]);
        uint32_t* f = reinterpret_cast<uint32_t*>(xr) + 3 * h;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            f[p] = hi[p];
            f[16 + p] = mi[p];
            f[32 + p] = lo[p];
        }
        uint2* b = reinterpret_cast<uint2*>(xr) + 3;  // chunk 1's half of part p: b[8 p]
        b[8 * h] = peb[0];
        b[16 - 8 * h] = peb[1];
#pragma unroll
        for (int t = 0; t < 3; ++t) reinterpret_cast<u32x4*>(xr)[2 + 4 * t + h] = pe[t];
        reinterpret_cast<u32x4*>(xr)[12 + h] = pe[3];
        if (h == 0) reinterpret_cast<u32x4*>(xr)[14] = pe[4];
    };

    int64_t grp = (int64_t)wv * gridDim.x + blockIdx.x;
    load_records(grp);
    stage_fwd_weights(sm, W);  // behind the first records' loads
    lookup();
    load_records(grp + stride);
    float v[12];  // the next group's colour: this lane's corners, a pair at a time
    {
        float w[12];
        Raw raw1[2][3];  // one round trip for both pairs
        fetch(0, raw);
        fetch(1, raw1);
        fetch_pe();
        weigh(0, raw, v);
        weigh(1, raw1, w);
#pragma unroll
        for (int c = 0; c < 12; ++c) v[c] += w[c];
        store_x(v);
    }
    __syncthreads();  // the weights; from here on the wavefronts run on their own
    const float b2a = W.b2[h], b2b = W.b2[2];

    for (; grp < ngroups; grp += stride) {
        const int64_t q0 = grp * GS;
        const bool alive = (nbits & kAliveW) != 0u;
        uint4 xb[8];  // this group's X fragments
        xb[0] = *xfirst;
#pragma unroll
        for (int t = 1; t < 8; ++t) xb[t] = xr[2 * t - 1 + h];
        {  // the backward's input row: X columns 0..39 (hi)
            uint4* row = rec.xrow + 5 * q0 + 5 * n;
            row[h] = xr[h];
            row[2 + h] = xr[2 + h];
            row[4] = xr[12];  // both halves, the same values
        }
        lookup();
        load_records(grp + 2 * stride);
        // A tile's MFMAs run in eight slots; the vector instructions of a slot
        // turn one pair of the tile before (relu, mask, split) into the next
        // layer's B fragments while the matrix core works, and every weight
        // fragment is read two steps ahead of its use.  The scheduling barriers
        // keep the compiler from gathering either kind together again.
        uint32_t mask0[2] = {0u, 0u}, mask1[2] = {0u, 0u};  // words 2h and 2h + 1 (T / 2)
        uint32_t h0[8][3][4];  // layer 1's B fragments [k-step][part][dword]
        uint32_t h1[2][2][4];  // layer 2's of a tile: [rows' half t, then samples' half s][part]
        f32x16 c, d;           // a tile in the making, the one before
        f32x4 lt[2], lg[2];    // samples 16s ..: the logits over a tile's features, over all before
        const f32x16 zero = {};
        auto pair0 = [&](int T, int j) {  // pair j (rows 2j, 2j + 1 of the lane) of tile T
            uint32_t(*f)[4] = h0[2 * T + (j >> 2)];
            split3(relu(d[2 * j]), relu(d[2 * j + 1]), f[0][j & 3], f[1][j & 3], f[2][j & 3]);
            mask_pair(f[0][j & 3], 8 * (T & 1) + j, mask0[T >> 1]);
            pin(f[0][j & 3], f[1][j & 3], f[2][j & 3], mask0[T >> 1]);
        };
        // the logits over tiles 0 .. T
        auto add_logits = [&](int T) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int o = 0; o < 3; ++o) lg[s][o] = T == 0 ? lt[s][o] : lg[s][o] + lt[s][o];
        };
        uint4 w2f;
        auto pair1 = [&](int T, int j) {
            uint32_t(*f)[4] = h1[j >> 2];
            split2(relu(d[2 * j]), relu(d[2 * j + 1]), f[0][j & 3], f[1][j & 3]);
            mask_pair(f[0][j & 3], 8 * (T & 1) + j, mask1[T >> 1]);
            pin(f[0][j & 3], f[1][j & 3], mask1[0], mask1[1]);
            if (j == 2 && T > 0) add_logits(T - 1);
            if (j == 5) w2f = w2p[16 * T];
            if (j >= 4) {
                // a lane's two groups of eight features (2h + t) to the four of one
                // sample half, a group to each 16 lanes
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const auto r = __builtin_amdgcn_permlane16_swap(h1[0][p][j & 3], h1[1][p][j & 3],
                                                                    false, false);
                    h1[0][p][j & 3] = r[0];
                    h1[1][p][j & 3] = r[1];
                }
            }
            if (j == 7) {  // layer 2 over the tile's 32 features
                const bf16x8 w = as_bf8(w2f);
                const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 2; ++s) lt[s] = mfma16x16x32(w, as_bf8(frag(h1[s][0])), z);
#pragma unroll
                for (int s = 0; s < 2; ++s) lt[s] = mfma16x16x32(w, as_bf8(frag(h1[s][1])), lt[s]);
            }
        };
        // ---- layer 0: H0^T = relu(W0^T X^T + b0) ----
        uint4 fa = w0b0[0], fb = w012[0], fc = w030[0];
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            if (T == 3) fetch(0, raw);  // the next group's inputs, from here to layer 1's end
            c = mfma32x32x16(fa, xb[0], zero);
            if (T > 0) pair0(T - 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            fa = w034[32 * T];
            c = mfma32x32x16(fb, xb[1], c);
            if (T > 0) pair0(T - 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            c = mfma32x32x16(fc, xb[2], c);
            if (T > 0) pair0(T - 1, 2);
            __builtin_amdgcn_sched_barrier(0);
            c = mfma32x32x16(fb, xb[3], c);
            if (T > 0) pair0(T - 1, 3);
            __builtin_amdgcn_sched_barrier(0);
            c = mfma32x32x16(fc, xb[4], c);
            if (T > 0) pair0(T - 1, 4);
            __builtin_amdgcn_sched_barrier(0);
            fc = w044[32 * T];
            c = mfma32x32x16(fb, xb[5], c);
            if (T > 0) pair0(T - 1, 5);
            __builtin_amdgcn_sched_barrier(0);
            fb = T < 3 ? w012[32 * (T + 1)] : w1p[64];
            c = mfma32x32x16(fa, xb[6], c);
            if (T > 0) pair0(T - 1, 6);
            __builtin_amdgcn_sched_barrier(0);
            fa = T < 3 ? w0b0[32 * (T + 1)] : w1p[0];
            c = mfma32x32x16(fc, xb[7], c);
            if (T > 0) pair0(T - 1, 7);
            __builtin_amdgcn_sched_barrier(0);
            if (T < 3) fc = w030[32 * (T + 1)];
            d = c;
        }
        // ---- layer 1: H1^T = relu(W1^T H0^T + b1); layer 2 over its tiles ----
        uint4 f[3] = {fa, fb};
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            // step 9T + k (the bias, then the k-steps) is in f[(9T + k) % 3]
            f[(9 * T + 2) % 3] = w1p[64 * (9 * T + 2)];
            if (T == 1) {
                weigh(0, raw, v);
                fetch(1, raw);
            }
            if (T == 3) {
                float w[12];
                weigh(1, raw, w);
#pragma unroll
                for (int i = 0; i < 12; ++i) v[i] += w[i];
                fetch_pe();
            }
            c = mfma32x32x16(f[(9 * T) % 3], sm.ones, zero);
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {  // 32 features: their hi parts, mid parts, lo parts
                const int s = 9 * T + 1 + 2 * kt;
                if (s + 2 < 36) f[(s + 2) % 3] = w1p[64 * (s + 2)];
#pragma unroll
                for (int m = 0; m < 6; ++m) {
                    c = mfma32x32x16(f[(s + (m & 1)) % 3], frag(h0[2 * kt + (m & 1)][m >> 1]), c);
                    if (m == 4 && s + 3 < 36) f[s % 3] = w1p[64 * (s + 3)];
                    if (m % 3 != 2) continue;
                    const int slot = 2 * kt + m / 3;
                    if (T > 0) {
                        pair1(T - 1, slot);
                    } else if (slot < 4) {  // the last layer-0 tile is k-steps 6 and 7's input
                        pair0(3, 2 * slot);
                        pair0(3, 2 * slot + 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            d = c;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) pair1(3, j);
        store_x(v);
        wave_lds_fence();
        add_logits(3);
        // ---- the masks and rgb ----
        {
            uint2* mw = reinterpret_cast<uint2*>(rec.relu + 8 * q0 + 8 * n + 2 * h);
            mw[0] = make_uint2(mask0[0], mask0[1]);
            mw[2] = make_uint2(mask1[0], mask1[1]);
            // the first 16 lanes hold both sample halves' logits: those of 16 .. 31 to the
            // lanes after them, then logit 1 to half 1; half h finishes channel h, half 0
            // channel 2 too (half 1 writes the unused fourth)
            uint32_t l[3];
#pragma unroll
            for (int o = 0; o < 3; ++o)
                l[o] = __builtin_amdgcn_permlane16_swap(__float_as_uint(lg[0][o]),
                                                        __float_as_uint(lg[1][o]), false, false)[0];
            const float x = __uint_as_float(
                __builtin_amdgcn_permlane32_swap(l[0], l[1], false, false)[0]);
            const float y = __uint_as_float(l[2]);
            const float a = sigmoidf_(x + b2a), b = sigmoidf_(y + b2b);
            float* rgb = reinterpret_cast<float*>(rec.rgb + q0) + 4 * n + h;
            rgb[0] = alive ? a : 0.f;
            rgb[2] = alive && h == 0 ? b : 0.f;
        }
    }
}

// ---- backward ----------------------------------------------------------------
// A workgroup takes rounds of four 32-record groups with four pairs of
// wavefronts, two wavefronts to a SIMD.  Of a pair, the gradient wavefront runs
// its group's chain
//   g_H1^T = W2 g_L^T (masked), g_H0^T = W1 g_H1^T (masked), g_X^T = W0[0:12] g_H0^T
// with the gradients as (hi, lo) pairs, in registers from end to end as in the
// forward: all rows are in layer 0's order.  The other, the weight wavefront, recomputes
//   H0^T = W0^T X^T + b0, H1 = H0 W1 + b1 under the forward's masks
// from hi parts (for the dW operands only; H1 comes out a feature to a lane, in
// layer 1's order, since its operands are the same fragments in the other order,
// and its mask bits out of LDS), adds its group's H1^T g_L to dW2, and
// then a slice of the whole round's dW1 += H0^T g_H1 (64 x 64) and dW0 += X^T g_H0
// (all inputs x 32).  Those contract over samples, so their operands cross
// wavefronts: H0, g_H1, g_H0 (hi) and X lie in LDS a row to a sample, and are read
// through the transposing LDS load, which hands a lane four samples of its
// feature.  W1 sits in LDS once: the gradient wavefronts read W1 rows out of the
// W1^T fragments with the same load.
//
// A round has two intervals, a barrier after each, so that one copy of the
// buffers will do:
//   1  weight: dW1 and dW0 of the round before      gradient: g_H1, a quarter of g_H0
//   2  weight: H0, H1, dW2                          gradient: stores, the rest
// Within a wavefront a tile is masked, split or relu'd pair by pair between the
// next tile's MFMAs.
//
// The rows' 8-byte pieces (four features) are permuted by the sample's index so
// that neither the stores (32 rows, one piece each) nor the transposing loads
// (four rows x 32 features to a wavefront half) meet in a bank.
//
// What bounds it: a round is 180 MFMAs of 32 cycles per SIMD and about as many
// cycles of vector work (1400 instructions of 4), which the two wavefronts overlap
// in part, and 40% of the time in the CU's LDS.
//
// Measured against eight wavefronts that shared one group (16 hidden features
// each, every product's operands through LDS on 16x16x32 MFMAs): 7.80M records
// 2632 -> 1232 us, 190k 98.2 -> 53.0 us, 24k 25.0 -> 15.0 us.  With relu of the
// recomputed activations in place of the forward's masks, which is not the same,
// 1144, 49.2 and 14.4 us; and at 7.80M records tiles split after their MFMAs instead
// of between the next one's cost 53 us more, db1 summed over lanes at each round (32
// registers fewer, three instructions a pair more) with the stores' and loads'
// addresses formed each time 175 us.
constexpr int kBwdPairs = 4;                   // wavefront pairs, a group each
constexpr int kBwdWaves = 2 * kBwdPairs;
constexpr int kRoundRec = kBwdPairs * GS;      // records of a round
constexpr int kFragPitch = 576, kHalfPitch = 288;  // W1^T fragments in LDS (16-bit values): lane
                                                   // halves 64 bytes, fragments 128 bytes of the
                                                   // 256-byte bank row apart
struct alignas(16) SmemBwd {
    uint16_t g1[kRoundRec * 128];   // g_H1, g_H0 and H0 (hi) by sample
    uint16_t g0[kRoundRec * 128];
    uint16_t h0[kRoundRec * 128];
    uint16_t x[kRoundRec * 40 + 24];  // X by sample; loads of columns 40..63 run into the next row
    uint4 w0[5 * 128];              // the forward image's W0^T chunks
    uint16_t w1[32 * kFragPitch];   // the forward image's W1^T fragments [row tile][k-step]
    uint2 w2[128];                  // W2's rows
    float b0[128], b1[128];
    uint4 w0g[8 * 2 * 12];          // W0[0:12] as g_X's A fragments [k-step][h][feature]
    uint16_t gl[kBwdPairs][3 * GS]; // dL/dlogit (hi) by logit
    uint32_t m1[kBwdPairs][4][GS];  // layer 1's ReLU mask words by word
};
static_assert(sizeof(SmemBwd) <= 160 * 1024, "a CU's LDS");

// Four samples of this lane's feature, from the pieces that the lane's group of
// 16 points at: lane i names row i / 4's piece i % 4 and receives column i.
__device__ __forceinline__ uint2 ld_tr(const void* p) {
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(p));
    return __builtin_bit_cast(uint2, v);
}
__device__ __forceinline__ uint4 ld_tr2(const void* p, const void* q) {
    const uint2 a = ld_tr(p), b = ld_tr(q);
    return make_uint4(a.x, a.y, b.x, b.y);
}

// sum over each half of the wavefront, in its last lane
__device__ __forceinline__ float half_sum(float x) {
    x += dpp_mov<kDppRowShr1>(x, 0.f);
    x += dpp_mov<kDppRowShr2>(x, 0.f);
    x += dpp_mov<kDppRowShr4>(x, 0.f);
    x += dpp_mov<kDppRowShr8>(x, 0.f);
    x += dpp_mov<kDppRowBcast15, 0xa>(x, 0.f);
    return x;
}

// x where bit k of m is set, else +0: the bit sign-extended by one v_bfe_i32
// and ANDed with x's bits (two instructions; a compare and a select take
// three, with the bit extraction)
__device__ __forceinline__ float keep_if(uint32_t m, int k, float x) {
    const uint32_t all = (uint32_t)__builtin_amdgcn_sbfe((int)m, k, 1);
    return __uint_as_float(__float_as_uint(x) & all);
}

__device__ __forceinline__ void stage_bwd_weights(SmemBwd& sm, const MlpPacked& W) {
    constexpr int NTH = 64 * kBwdWaves;
    const int tid = threadIdx.x;
    for (int e = tid; e < 5 * 128; e += NTH) sm.w0[e] = W.fwd[e];
    const uint4* img = W.fwd + kImgW1 / 8;  // [row tile][9 steps, the first the bias][lane]
#pragma unroll
    for (int k = 0; k < 32 * 64 / NTH; ++k) {
        const int e = tid + NTH * k, f = e >> 6, l = e & 63;
        *reinterpret_cast<uint4*>(sm.w1 + f * kFragPitch + (l >> 5) * kHalfPitch + 8 * (l & 31)) =
            img[((f >> 3) * 9 + 1 + (f & 7)) * 64 + l];
    }
    if (tid < 128) {
        sm.w2[tid] = *reinterpret_cast<const uint2*>(W.w2 + 32 * tid);  // w0 w1 | w2 0
        sm.b0[tid] = W.b0[tid];
        sm.b1[tid] = W.b1[tid];
    } else if (tid < 128 + 8 * 2 * 12) {
        const int e = tid - 128, m = e % 12, h = (e / 12) & 1, ks = e / 24;
        sm.w0g[e] = *reinterpret_cast<const uint4*>(W.w0 + 128 * m + 16 * ks + 8 * h);
    }
}

__global__ void __launch_bounds__(64 * kBwdWaves) k_mlp_bwd(StepParams P, MlpPacked W,
                                                            RayBuffers R, Records rec,
                                                            float* __restrict__ dw_partial) {
    __shared__ SmemBwd sm;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int w = wv & (kBwdPairs - 1);  // the group of the round
    const int lane = lane_id(), n = lane & 31, h = lane >> 5;
    const int64_t total = min((int64_t)R.total[0], P.capacity);
    const int64_t nrounds = (total + kRoundRec - 1) / kRoundRec;
    const int64_t r0 = blockIdx.x, stride = gridDim.x;
    float* const out = dw_partial + (int64_t)blockIdx.x * kPartStride;
    float* const red = reinterpret_cast<float*>(sm.g1);  // the last reductions' room
    constexpr int kRedDb1 = 4 * 384, kRedDb2 = kRedDb1 + 4 * 128;  // after dW2's [4][384]
    stage_bwd_weights(sm, W);
    // where this lane's sample stores its pieces, and what it points the
    // transposing loads at: row rr (+ 4h + 8jj + 16t) and piece pc of 16 c16 features
    const int rr = (lane & 15) >> 2, pc = lane & 3, c16 = (lane >> 4) & 1;
    // the bytes of this lane's first piece in its sample's row: piece
    // 8T + 4 (q / 2) + 2h + q % 2, which holds the lane's rows 8q + 4h .. of tile T (layer
    // 0's order), lies at the same offset ^ (64 T + 32 (q / 2) + 8 (q % 2)).  Anew in each
    // round: as loop invariants the sixteen addresses would take as many registers
    auto row_at = [&]() {
        uint32_t at = 256 * (GS * w + n) + 8 * ((((n & 3) << 3) | (n >> 2)) ^ (2 * h));
        asm volatile("" : "+v"(at));
        return at;
    };
    auto piece = [](uint16_t* rows, uint32_t at, int T, int q) {
        return reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(rows) +
                                        (at ^ (64u * T + 32u * (q >> 1) + 8u * (q & 1))));
    };

    if (wv >= kBwdPairs) {
        // ---- the gradient chain ----
        float4 adj, nadj;
        uint2 mk0, nmk0, nmk1;  // this lane half's ReLU mask words of the two layers
        uint32_t bits, nbits;
        auto load = [&](int64_t rnd) {  // the next round's
            const int64_t q = rnd * kRoundRec + GS * w + n;
            nadj = make_float4(0.f, 0.f, 0.f, 0.f);
            nmk0 = nmk1 = make_uint2(0u, 0u);
            nbits = 0u;
            if (q < total) {
                nadj = rec.adj[q];
                nbits = __float_as_uint(rec.ab[q].y);
                nmk0 = reinterpret_cast<const uint2*>(rec.relu)[4 * q + h];
                nmk1 = reinterpret_cast<const uint2*>(rec.relu)[4 * q + 2 + h];
            }
        };
        float db1[64], db2[3] = {0.f, 0.f, 0.f};  // this lane's sample of each round
#pragma unroll
        for (int i = 0; i < 64; ++i) db1[i] = 0.f;
        // W1 rows (in layer 0's order) out of the W1^T fragments
        const uint16_t* const wa = sm.w1 + c16 * kFragPitch + (pc & 1) * kHalfPitch +
                                   8 * (16 * h + rr) + 4 * (pc >> 1);
        const uint4* const w0p = sm.w0g + 12 * h + (n < 12 ? n : 0);
        const f32x16 zero = {};
        uint32_t gh[8][4], glo[8][4];  // g_H1's B fragments [k-step][dword], hi and lo
        f32x16 gx;
        f32x16 d;                      // a finished tile, split while the next one's MFMAs run
        float va, vb;
        // pair j (rows 2j, 2j + 1 of the lane) of tile T in two steps: masked, then split
        auto mask_of = [&](uint32_t m, int p, int j) {
            va = keep_if(m, p, d[2 * j]);
            vb = keep_if(m, 16 + p, d[2 * j + 1]);
        };
        auto mask0 = [&](int T, int j) { mask_of(T & 2 ? mk0.y : mk0.x, 8 * (T & 1) + j, j); };
        // g_H1's rows are in layer 0's order: feature 16 (j / 4) + 8h + .. of the tile is the
        // forward's row pair 4h + j % 4 of lane half j / 4
        uint32_t mk1[2];
        auto mask1 = [&](int T, int j) {
            if (j == 0 && !(T & 1))
#pragma unroll
                for (int f = 0; f < 2; ++f) mk1[f] = sm.m1[w][2 * f + (T >> 1)][n] >> (4 * h);
            mask_of(mk1[j >> 2], 8 * (T & 1) + (j & 3), j);
        };
        auto w1 = [&](int T, int ks) {
            const uint16_t* a = wa + ((ks >> 1) * 8 + 2 * T) * kFragPitch + 32 * (ks & 1);
            return ld_tr2(a, a + 64);
        };
        // pair j of g_H1's tile T: gh, glo and db1
        auto pair1 = [&](int T, int j) {
            mask1(T, j);
            db1[16 * T + 2 * j] += va;
            db1[16 * T + 2 * j + 1] += vb;
            uint32_t &hi = gh[2 * T + (j >> 2)][j & 3], &lo = glo[2 * T + (j >> 2)][j & 3];
            split2(va, vb, hi, lo);
            // here, not at the round's end with va and vb alive till then
            asm volatile("" : "+v"(db1[16 * T + 2 * j]), "+v"(db1[16 * T + 2 * j + 1]), "+v"(hi), "+v"(lo));
        };
        uint32_t hi[8], lo[8];  // g_H0's pairs of a tile
        // layer 0's features of tile T into the records' gradients
        auto add_gx = [&](int T) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {  // the hi parts, then the lo parts
                const uint32_t* v = p ? lo : hi;
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    gx = mfma32x32x16(w0p[24 * (2 * T + t)],
                                      make_uint4(v[4 * t], v[4 * t + 1], v[4 * t + 2], v[4 * t + 3]), gx);
            }
        };
        auto pair0_split = [&](int j) {
            split2(va, vb, hi[j], lo[j]);
            asm volatile("" : "+v"(hi[j]), "+v"(lo[j]));
        };
        load(r0);
        __syncthreads();  // the weights
        for (int64_t rnd = r0; rnd < nrounds; rnd += stride) {
            // ---- interval 1 ----
            adj = nadj;
            bits = nbits;
            mk0 = nmk0;
            sm.m1[w][2 * h][n] = nmk1.x;
            sm.m1[w][2 * h + 1][n] = nmk1.y;
            wave_lds_fence();  // this wavefront reads both halves'
            {
                uint32_t h01, l01, h2, l2;
                split2(adj.x, adj.y, h01, l01);
                split2(adj.z, 0.f, h2, l2);
                db2[0] += adj.x;
                db2[1] += adj.y;
                db2[2] += adj.z;
                if (h == 0) {
                    uint16_t* g = &sm.gl[w][n];
                    g[0] = (uint16_t)(h01 & 0xffffu);
                    g[GS] = (uint16_t)(h01 >> 16);
                    g[2 * GS] = (uint16_t)h2;
                }
                // the hi parts in half 0's k, the lo parts in half 1's
                const uint4 b = make_uint4(h ? l01 : h01, h ? l2 : h2, 0u, 0u);
                auto w2 = [&](int T) {
                    const uint2 f = sm.w2[32 * T + mlp_feature(0, n)];
                    return make_uint4(f.x, f.y, 0u, 0u);
                };
                // g_H1 a tile at a time, each followed by its k-steps of g_H0's first tile
                // under the next one's split
                f32x16 e = mfma32x32x16(w2(0), b, zero), c;
#pragma unroll
                for (int T = 0; T < 5; ++T) {
                    uint4 f0, f1;
                    d = e;
                    if (T < 3) e = mfma32x32x16(w2(T + 1), b, zero);
                    if (T > 0) {
                        f0 = w1(0, 2 * T - 2);
                        f1 = w1(0, 2 * T - 1);
                    }
                    if (T < 4) {
                        pair1(T, 0);
                        pair1(T, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (T > 0) {
                            const int ks = 2 * T - 2 + (k & 1);
                            c = mfma32x32x16(k & 1 ? f1 : f0, frag(k < 2 ? gh[ks] : glo[ks]),
                                             T == 1 && k == 0 ? zero : c);
                        }
                        if (T < 4) {
                            pair1(T, 2 + k);
                            if (k == 3) pair1(T, 6);
                            if (k == 3) pair1(T, 7);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                d = c;
            }
            __syncthreads();
            // ---- interval 2 ----
            load(rnd + stride);
            const uint32_t at = row_at();
            gx = zero;
            uint4 f[3] = {w1(1, 0), w1(1, 1)};  // step k is in f[k % 3]
#pragma unroll
            for (int T = 1; T < 4; ++T) {
                f32x16 c = zero;
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) {  // 32 features: their hi parts, their lo parts
                    const int k = 8 * (T - 1) + 2 * kt;
                    if (k < 22) f[(k + 2) % 3] = w1(1 + (k + 2) / 8, (k + 2) & 7);
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const int ks = 2 * kt + (m & 1), j = 2 * kt + (m >> 1);
                        c = mfma32x32x16(f[(k + (m & 1)) % 3], frag(m < 2 ? gh[ks] : glo[ks]), c);
                        if (m == 2 && k < 22) f[k % 3] = w1(1 + (k + 3) / 8, (k + 3) & 7);
                        if (m & 1) {
                            pair0_split(j);
                            if (j & 1) *piece(sm.g0, at, T - 1, j >> 1) = make_uint2(hi[j - 1], hi[j]);
                        } else {
                            mask0(T - 1, j);
                            if (T == 1 && m == 2)  // g_H1's rows, between the first MFMAs
#pragma unroll
                                for (int q = 0; q < 4; ++q) {
                                    const uint32_t* g = gh[j - 1 + (q >> 1)] + 2 * (q & 1);
                                    *piece(sm.g1, at, j >> 1, q) = make_uint2(g[0], g[1]);
                                }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                add_gx(T - 1);
                d = c;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                mask0(3, j);
                pair0_split(j);
                if (j & 1) *piece(sm.g0, at, 3, j >> 1) = make_uint2(hi[j - 1], hi[j]);
            }
            add_gx(3);
            // the record's gradient row: lane half h holds features 4h .. 4h + 3
            // and, half 0, 8 .. 11; half 1 adds dL/dsigma
            const int64_t q = rnd * kRoundRec + GS * w + n;
            if (q < total) {
                const bool on = (bits & kAliveW) != 0u;
                float4* row = rec.grad + 4 * q + h;
                row[0] = on ? make_float4(gx[0], gx[1], gx[2], gx[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
                row[2] = h ? make_float4(adj.w, 0.f, 0.f, 0.f)
                           : on ? make_float4(gx[4], gx[5], gx[6], gx[7]) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            __syncthreads();
        }
        __syncthreads();  // the weight wavefronts have read the last round's buffers
        // db1 and db2: each wavefront's samples, then the four wavefronts'
#pragma unroll
        for (int i = 0; i < 64; ++i) {
            const float v = half_sum(db1[i]);
            if (n == 31)
                red[kRedDb1 + 128 * w + 32 * (i >> 4) + 16 * ((i >> 3) & 1) + 8 * h + (i & 7)] = v;
        }
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            const float v = half_sum(db2[o]);
            if (lane == 31) red[kRedDb2 + 4 * w + o] = v;
        }
    } else {
        // ---- the weights ----
        f32x16 dW1[2][2], dW0[2];
        f32x4 dW2[4];
        const f32x16 zero = {};
#pragma unroll
        for (int a = 0; a < 2; ++a) dW1[a][0] = dW1[a][1] = dW0[a] = zero;
#pragma unroll
        for (int T = 0; T < 4; ++T) dW2[T] = f32x4{0.f, 0.f, 0.f, 0.f};
        uint4 xb[3];  // the group's X fragments: columns 8h, 16 + 8h, and 32 (h = 1: zeros)
        uint2 m0;     // layer 0's ReLU mask words of this lane half
        auto load = [&](int64_t rnd) {
            const int64_t q = rnd * kRoundRec + GS * w + n;
            xb[0] = xb[1] = xb[2] = make_uint4(0u, 0u, 0u, 0u);
            m0 = make_uint2(0u, 0u);
            if (q < total) {
                const uint4* row = rec.xrow + 5 * q;
                xb[0] = row[h];
                xb[1] = row[2 + h];
                if (h == 0) xb[2] = row[4];
                m0 = reinterpret_cast<const uint2*>(rec.relu)[4 * q + h];
            }
        };
        const uint4* const w0p = sm.w0 + 128 * h + n;
        const float* const b0p = sm.b0 + 8 * h;
        const uint16_t* const w1p = sm.w1 + h * kHalfPitch + 8 * n;
        // layer 1: the bias of this lane's feature of tile 0, and where its mask bits are
        const float* const b1p = sm.b1 + mlp_feature(1, n);
        const int bit1 = 16 * (n & 1) + 2 * (n >> 3) + ((n >> 1) & 1);
        const uint32_t* const m1p = &sm.m1[w][2 * ((n >> 2) & 1)][4 * h];
        // dW1 and dW0 of the round in the buffers
        auto dw = [&]() {
            uint4 fr[2][7];  // a k-step's operands, read one step ahead
            // bytes from a group's first row: [feature tile][t][jj], and X's
            uint32_t fa[5][2][2], xa;
            {
                int ro = rr, po = 4 * c16 + pc;
                asm volatile("" : "+v"(ro), "+v"(po));  // anew in each round, like row_at
                const int tile[5] = {2 * (w & 1), 2 * (w & 1) + 1, 2 * (w >> 1), 2 * (w >> 1) + 1, w};
#pragma unroll
                for (int f = 0; f < 5; ++f)
#pragma unroll
                    for (int tj = 0; tj < 4; ++tj)  // row 16 t + 8 jj + 4 h + rr, piece 8 T + po, swizzled
                        fa[f][tj >> 1][tj & 1] = 256u * (8 * tj + 4 * h + ro) + 64u * (tile[f] ^ ro) +
                                                 8u * (po ^ (2 * tj + h));
                xa = 80u * (4 * h + ro) + 8u * po;
            }
            auto rd = [&](int g, int t, uint4 (&f)[7]) {
                auto feat = [&](const uint16_t* rows, int i) {
                    const uint8_t* b = reinterpret_cast<const uint8_t*>(rows + GS * 128 * g);
                    return ld_tr2(b + fa[i][t][0], b + fa[i][t][1]);
                };
                f[0] = feat(sm.h0, 0);
                f[2] = feat(sm.g1, 2);
                f[1] = feat(sm.h0, 1);
                f[3] = feat(sm.g1, 3);
                const uint8_t* x = reinterpret_cast<const uint8_t*>(sm.x + 40 * (GS * g + 16 * t)) + xa;
                f[4] = ld_tr2(x, x + 8 * 80);
                f[6] = feat(sm.g0, 4);
                f[5] = ld_tr2(x + 64, x + 64 + 8 * 80);
            };
            rd(0, 0, fr[0]);
#pragma unroll
            for (int g = 0; g < kBwdPairs; ++g)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const uint4(&f)[7] = fr[t];
                    if (t == 0)
                        rd(g, 1, fr[1]);
                    else if (g + 1 < kBwdPairs)
                        rd(g + 1, 0, fr[0]);
                    dW1[0][0] = mfma32x32x16(f[0], f[2], dW1[0][0]);
                    dW1[1][0] = mfma32x32x16(f[1], f[2], dW1[1][0]);
                    dW1[0][1] = mfma32x32x16(f[0], f[3], dW1[0][1]);
                    dW1[1][1] = mfma32x32x16(f[1], f[3], dW1[1][1]);
                    dW0[0] = mfma32x32x16(f[4], f[6], dW0[0]);
                    dW0[1] = mfma32x32x16(f[5], f[6], dW0[1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
        };
        load(r0);
        __syncthreads();  // the weights
        for (int64_t rnd = r0; rnd < nrounds; rnd += stride) {
            // ---- interval 1 ----
            if (rnd != r0) dw();
            __syncthreads();
            // ---- interval 2 ----
            {
                uint4* xr = reinterpret_cast<uint4*>(sm.x + (GS * w + n) * 40);
                xr[h] = xb[0];
                xr[2 + h] = xb[1];
                if (h == 0) xr[4] = xb[2];
            }
            uint32_t h0[8][4];
            const uint32_t at = row_at();
            f32x16 c, d;  // a tile in the making, the one before
            // masked by the forward's bits, not by these values' signs
            auto pair0 = [&](int T, int j, uint32_t m) {
                uint32_t* f = h0[2 * T + (j >> 2)];
                const int p = 8 * (T & 1) + j;
                f[j & 3] = pk_bf(keep_if(m, p, d[2 * j]), keep_if(m, 16 + p, d[2 * j + 1]));
                if (j & 1) *piece(sm.h0, at, T, j >> 1) = make_uint2(f[(j & 3) - 1], f[j & 3]);
            };
#pragma unroll
            for (int T = 0; T < 4; ++T) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {  // the accumulators start at the bias
                    const float4 b = *reinterpret_cast<const float4*>(b0p + 32 * T + 16 * (q >> 1) + 4 * (q & 1));
                    c[4 * q] = b.x;
                    c[4 * q + 1] = b.y;
                    c[4 * q + 2] = b.z;
                    c[4 * q + 3] = b.w;
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    // h = 1's last chunk meets zeros
                    c = mfma32x32x16(w0p[(k < 2 ? 256 * k : 512 - 128 * h) + 32 * T], xb[k], c);
                    if (T > 0) {
                        const uint32_t m = (T - 1) & 2 ? m0.y : m0.x;
                        pair0(T - 1, 3 * k, m);
                        pair0(T - 1, 3 * k + 1, m);
                        if (k < 2) pair0(T - 1, 3 * k + 2, m);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                d = c;
            }
            const uint32_t m0_3 = m0.y;
            load(rnd + stride);
            uint2 gl[4];  // dL/dlogit (lane & 3; the fourth's sums go unused) of samples 8q + 4h ..
#pragma unroll
            for (int q = 0; q < 4; ++q)
                gl[q] = *reinterpret_cast<const uint2*>(&sm.gl[w][GS * min(lane & 3, 2) + 8 * q + 4 * h]);
            auto w1 = [&](int k) { return *reinterpret_cast<const uint4*>(w1p + k * kFragPitch); };
            uint4 f1[3] = {w1(0), w1(1)};  // read two steps ahead
            uint32_t r[2];
            uint4 m1[4];  // the mask words of this lane's samples 8q + 4h ..
            auto pair1 = [&](int T, int j) {
                if (j == 0 && !(T & 1))
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        m1[q] = *reinterpret_cast<const uint4*>(m1p + GS * (T >> 1) + 8 * q);
                const uint4& m = m1[j >> 1];
                const int b = bit1 + 8 * (T & 1);
                r[j & 1] = pk_bf(keep_if(j & 1 ? m.z : m.x, b, d[2 * j]),
                                 keep_if(j & 1 ? m.w : m.y, b, d[2 * j + 1]));
                if (j & 1) dW2[T] = mfma4x4x4(gl[j >> 1].x, gl[j >> 1].y, r[0], r[1], dW2[T]);
            };
#pragma unroll
            for (int T = 0; T < 4; ++T) {
                const float b1 = b1p[32 * T];
#pragma unroll
                for (int i = 0; i < 16; ++i) c[i] = b1;
#pragma unroll
                for (int ks = 0; ks < 8; ++ks) {
                    const int k = 8 * T + ks;
                    if (k < 30) f1[(k + 2) % 3] = w1(k + 2);
                    c = mfma32x32x16(frag(h0[ks]), f1[k % 3], c);
                    if (T > 0)
                        pair1(T - 1, ks);
                    else if (ks < 4) {  // the last layer-0 tile is k-steps 6 and 7's input
                        pair0(3, 2 * ks, m0_3);
                        pair0(3, 2 * ks + 1, m0_3);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                d = c;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) pair1(3, j);
            __syncthreads();
        }
        if ((int)blockIdx.x < (int)nrounds) dw();
        __syncthreads();  // the buffers are free for the reductions
        int f1 = n;
        asm volatile("" : "+v"(f1));  // not a register through the loop
        f1 = mlp_feature(1, f1);
#pragma unroll
        for (int T = 0; T < 4; ++T)
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                const float v = dW2[T][o] + __shfl_xor(dW2[T][o], 32, 64);
                if (h == 0) red[384 * w + 3 * (32 * T + f1) + o] = v;
            }
        // ---- this workgroup's dW partial ----
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int in = 32 * a + 8 * (i >> 2) + 4 * h + (i & 3);
                out[kW1 + (64 * (w & 1) + in) * 128 + 64 * (w >> 1) + n] = dW1[a][0][i];
                out[kW1 + (64 * (w & 1) + in) * 128 + 64 * (w >> 1) + 32 + n] = dW1[a][1][i];
                if (in < 39)
                    out[kW0 + in * 128 + 32 * w + n] = dW0[a][i];
                else if (in == 39)
                    out[kB0 + 32 * w + n] = dW0[a][i];
            }
    }
    __syncthreads();
    const int tid = threadIdx.x;
    if (tid < 384) {
        out[kW2 + tid] = ((red[tid] + red[384 + tid]) + red[768 + tid]) + red[1152 + tid];
    } else {
        const float* d = red + kRedDb1 + (tid - 384);
        out[kB1 + tid - 384] = ((d[0] + d[128]) + d[256]) + d[384];
    }
    if (tid < 3) {
        const float* d = red + kRedDb2 + tid;
        out[kB2 + tid] = ((d[0] + d[4]) + d[8]) + d[12];
    }
}

// Sum of the per-workgroup dW partials (dw_reduce_block): one workgroup per
// kReduceVec four-parameter vectors.  The fused step runs these workgroups
// inside the scatter's launch instead (launch_scatter), where they overlap the
// scatter's atomics; this launch serves the optimizer-only step.
__global__ void __launch_bounds__(256) k_dw_reduce(const float* __restrict__ part, int nparts,
                                                   float* __restrict__ dw, MlpAdam A) {
    __shared__ float4 red[kReduceGrp * kReduceVec];
    dw_reduce_block(blockIdx.x, part, nparts, dw, A, red);
}


}  // namespace

namespace pvdb {



int launch_mlp(bool bwd, bool bf16col, int grid, const StepParams& P, const TopoView& t,
               const void* color, const MlpPacked& W, const RayBuffers& R, const Records& rec,
               float* dw_partial, hipStream_t s) {
    if (bwd) {
        hipLaunchKernelGGL(k_mlp_bwd, dim3(grid), dim3(64 * kBwdWaves), 0, s, P, W, R, rec,
                           dw_partial);
        PVDB_LAUNCHED("k_mlp_bwd");
    } else {
        const auto kernel = bf16col ? k_mlp_fwd<true> : k_mlp_fwd<false>;
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * kFwdWaves), 0, s, P, t, color, W, R, rec);
        PVDB_LAUNCHED("k_mlp_fwd");
    }
    return PVDB_OK;
}

int launch_dw_reduce(const float* part, int nparts, float* dw, const MlpAdam& adam,
                     hipStream_t s) {
    hipLaunchKernelGGL(k_dw_reduce, dim3(kReduceBlocks), dim3(256), 0, s, part, nparts, dw, adam);
    PVDB_LAUNCHED("k_dw_reduce");
    return PVDB_OK;
}


}  // namespace pvdb
