// Fused step, sample side: the view-dependent RGB MLP (39-128-128-3, ReLU,
// sigmoid; plenvdb/lib/dvgo.py:91-109,354-362) on MFMA, forward and backward,
// over groups of 32 consecutive records (two 16-sample MFMA tiles).
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
// k_mlp_fwd gathers the colour features and writes each record's rgb, ReLU masks
// and bf16 input row (so the backward reads 80 bytes per record instead of
// redoing 8 gathers).  k_mlp_bwd recomputes H0 and H1 (for the dW operands) in
// wavefronts that own a slice of the hidden features each and exchange
// activations through LDS, takes each sample's dL/dlogit and dL/dsigma from
// the composite pass, runs g_H1^T = W2 g_L^T, g_H0^T = W1 g_H1^T (masked by
// the ReLUs, kept as bit masks), g_X^T = W0[0:12] g_H0^T, accumulates dW over
// each group's 32 samples (K = 32) in registers (one partial per workgroup),
// and writes each record's feature and sigma gradients; the scatter
// (fused_scatter.hip) then adds them to the grids with the "leaf must exist"
// rule (densityvdb.cu:16-27, colorvdb.cu:28-37).  Both kernels load a group's
// records into registers while the previous group computes.

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

constexpr int GS = 32;       // records per group
constexpr int NT = GS / 16;  // 16-sample MFMA tiles per group
constexpr int XM = 72;       // sample-major stride of X (64 + 8)
constexpr int SM = 136;      // sample-major stride of 128-wide activations (128 + 8)
constexpr int GM = 24;       // sample-major stride of dL/dlogit (16 + 8)
constexpr int FM = 40;       // feature-major stride (32 samples + 8; rows 16-byte aligned)
constexpr int XF_ROWS = 48;  // feature-major X rows: inputs 0..39 are used

__device__ __forceinline__ bf16x8 ld_frag(const uint16_t* p) {  // 16-byte aligned
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ s16x4 ld_frag4(const uint16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return __builtin_bit_cast(s16x4, v);
}

__device__ __forceinline__ bf16x8 as_bf8(const uint4& v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ void split_bf(float x, uint16_t& h, uint16_t& l) {
    uint32_t hh, ll;
    split2(x, 0.f, hh, ll);
    h = (uint16_t)hh;
    l = (uint16_t)ll;
}

// DPP permutation within rows (quad permutes, the half-row mirror), all lanes
// active: every lane reads a valid source, so the move needs no old value
// (update_dpp's would be materialised with a v_mov).
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
}

// A lane holds four consecutive features (rows) of one sample; the four lanes of
// a quad hold four consecutive samples.  Returns row (lane & 3) of the quad's
// four samples, as four bf16 in two dwords: two quad swaps instead of four
// 2-byte stores per lane.
__device__ __forceinline__ uint2 quad_transpose(uint2 h, int q) {
    const uint32_t v0 = h.x & 0xffffu, v1 = h.x >> 16, v2 = h.y & 0xffffu, v3 = h.y >> 16;
    // exchange 1 (lanes q, q^1): even lanes gather rows 0/2, odd lanes rows 1/3, of the pair
    const uint32_t send = (q & 1) ? (v0 | (v2 << 16)) : (v1 | (v3 << 16));
    const uint32_t recv = dpp<0xB1>(send);  // quad_perm [1,0,3,2]
    const uint32_t A = (q & 1) ? ((recv & 0xffffu) | (v1 << 16)) : (v0 | (recv << 16));
    const uint32_t B = (q & 1) ? ((recv >> 16) | (v3 << 16)) : (v2 | (recv & 0xffff0000u));
    // exchange 2 (lanes q, q^2): rows (q & 1) and (q & 1) + 2 of the two pairs
    const uint32_t send2 = (q & 2) ? A : B;
    const uint32_t recv2 = dpp<0x4E>(send2);  // quad_perm [2,3,0,1]
    return (q & 2) ? make_uint2(recv2, B) : make_uint2(A, recv2);
}

// Four consecutive features fr..fr+3 of sample `col`: sample-major (hi, lo)
// pairs into sh/sl, and (FMC) the hi parts feature-major into fm.
template <bool FMC>
__device__ __forceinline__ void st_act(uint16_t* sh, uint16_t* sl, uint16_t* fm, int col, int fr,
                                       int lane, const float* v) {
    uint2 hi, lo;
    split2(v[0], v[1], hi.x, lo.x);
    split2(v[2], v[3], hi.y, lo.y);
    *reinterpret_cast<uint2*>(&sh[col * SM + fr]) = hi;
    *reinterpret_cast<uint2*>(&sl[col * SM + fr]) = lo;
    if constexpr (FMC) {
        const int q = lane & 3;
        *reinterpret_cast<uint2*>(&fm[(fr + q) * FM + (col & ~3)]) = quad_transpose(hi, q);
    }
}

// The hi parts of four consecutive features fr..fr+3 of sample `col`:
// sample-major into sh and feature-major into fm.
__device__ __forceinline__ void st_hi_fm(uint16_t* sh, uint16_t* fm, int col, int fr, int lane,
                                         const float* v) {
    uint2 hi, lo;
    split2(v[0], v[1], hi.x, lo.x);
    split2(v[2], v[3], hi.y, lo.y);
    *reinterpret_cast<uint2*>(&sh[col * SM + fr]) = hi;
    const int q = lane & 3;
    *reinterpret_cast<uint2*>(&fm[(fr + q) * FM + (col & ~3)]) = quad_transpose(hi, q);
}

// The hi parts of four consecutive features fr..fr+3 of sample `col`,
// feature-major into fm (the feature-major half of st_act<true>).
__device__ __forceinline__ void st_fm(uint16_t* fm, int col, int fr, int lane, const float* v) {
    uint2 hi, lo;
    split2(v[0], v[1], hi.x, lo.x);
    split2(v[2], v[3], hi.y, lo.y);
    const int q = lane & 3;
    *reinterpret_cast<uint2*>(&fm[(fr + q) * FM + (col & ~3)]) = quad_transpose(hi, q);
}

// a (bf16 weight) times a split activation
__device__ __forceinline__ f32x4 mfma_w(const bf16x8& a, const bf16x8& bh, const bf16x8& bl,
                                        f32x4 c) {
    c = mfma16x16x32(a, bh, c);
    return mfma16x16x32(a, bl, c);
}

// dW products (activation x gradient) use the hi parts only, and the backward
// recomputes the activations they take from hi parts: the sums over a step's
// samples average that rounding (a device check keeps every MLP gradient
// within 6e-4 of FP64), so the gradients' lo parts stay sample-major.

// x where bit k of m is set, else +0: the bit sign-extended by one v_bfe_i32
// and ANDed with x's bits (two instructions; a compare and a select take
// three, with the bit extraction)
__device__ __forceinline__ float keep_if(uint32_t m, int k, float x) {
    const uint32_t all = (uint32_t)__builtin_amdgcn_sbfe((int)m, k, 1);
    return __uint_as_float(__float_as_uint(x) & all);
}

// ---- forward -----------------------------------------------------------------
// A wavefront takes a group of 32 records through the whole network by itself:
// its activations never leave its registers, so there is no barrier and no
// exchange between wavefronts once the weights are in LDS.  The D fragment of
// v_mfma_f32_32x32x16_bf16 (lane (h, n), h = lane / 32: features
// 32T + 8q + 4h + i of sample n, q, i < 4) is the next layer's B fragment when
// that layer's weights are stored with their K index permuted to match:
// position 8h + j of k-step 2T + t stands for feature
// 32T + 16t + 8 (j / 4) + 4h + j % 4.  A weight fragment read from LDS (8 LDS
// cycles) covers the three parts of the split activations: 96 cycles of its
// SIMD's matrix core.  X and H0 enter their products as (hi, mid, lo) triples,
// so the pre-activations, and with them the ReLU masks the backward applies,
// carry fp32 precision; H1 enters the logits as (hi, lo) pairs.
//
// X has 40 columns (12 features, 27 encoding inputs, the bias input) in three
// parts.  Stacked along K they are 15 chunks of 8 columns, two to a k-step, in
// the order
//   hi A, hi B | mid A, mid B | lo A, lo B | hi 2, hi 3 | hi 4, mid 2 |
//   mid 3, mid 4 | lo 2, lo 3 | lo 4, ones
// where chunk A is features 0..7, B features 8..11 and columns 12..15, and
// 2..4 columns 8c..8c + 7; they sit in a tile of the wavefront's own in LDS.
// The ones meet b0's own split, so the accumulators start at zero.
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
// (and 32 of 8) and about 1150 vector instructions of 4 cycles; two wavefronts
// per SIMD (250 registers) overlap them in part.  32x32x16 MFMAs are half as many
// to issue as 16x16x32 ones.  The splits stay an unpacking and a subtraction:
// a dot-product instruction does both at once, but runs on the matrix core
// and does not overlap with MFMAs.  The logits, 3 of 32 rows, use 4x4x4 MFMAs.
//
// Measured against four wavefronts that shared a group (32 hidden features each,
// activations exchanged through LDS, three barriers a group): 7.80M records with
// bf16 colour 2029 -> 982 us, 190k with fp32 colour 61.4 -> 36.8 us; 24k, one
// group to a wavefront, 13.8 -> 14.8 us.  On 16x16x32 MFMAs 1204 us.  With the
// gather in the march (features through memory) 900 us, and the march 485 us
// instead of 224.
constexpr int kFwdWaves = 4;
constexpr int kXChunks = 15;
struct alignas(16) SmemFwd {
    uint4 w0[6 * 128];             // [chunk][hidden feature]: W0^T columns 8c .. 8c + 7; b0's split
    uint4 w1[4 * 9 * 64];          // [row tile][step][lane]: b1's split, then W1^T's A
                                   // fragments of the eight k-steps, K permuted
    uint4 w2[8 * 2 * 4];           // W2^T rows [k-step][h][logit, zeros], K permuted
    uint4 ones[2];                 // [h] the inputs that the biases' splits are multiplied with
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
    const uint4* const xlast = h ? &sm.ones[0] : &xr[14];
    // W0 fragments: this lane's rows of the k-steps' chunk pairs (A, B), (2, 3),
    // (4, 2), (3, 4) and (4, bias)
    const uint4* const w0ab = sm.w0 + 128 * h + n;
    const uint4* const w023 = sm.w0 + 128 * (2 + h) + n;
    const uint4* const w042 = sm.w0 + 128 * (4 - 2 * h) + n;
    const uint4* const w034 = sm.w0 + 128 * (3 + h) + n;
    const uint4* const w04b = sm.w0 + 128 * (4 + h) + n;
    const uint4* const w1p = sm.w1 + lane;
    const uint4* const w2p = sm.w2 + 4 * h + (n & 3);

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
        pe[1] = row[3 + 2 * h];
        pe[2] = row[6 + h];
        pe[3] = row[9 + h];
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
            f[8 + p] = mi[p];
            f[16 + p] = lo[p];
        }
        uint2* b = reinterpret_cast<uint2*>(xr) + 3;  // chunk B's half of part p: b[4 p]
        b[4 * h] = peb[0];
        b[8 - 4 * h] = peb[1];
#pragma unroll
        for (int t = 0; t < 4; ++t) reinterpret_cast<u32x4*>(xr)[6 + 2 * t + h] = pe[t];
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
#pragma unroll
        for (int t = 0; t < 7; ++t) xb[t] = xr[2 * t + h];
        xb[7] = *xlast;
        {  // the backward's input row: X columns 0..39 (hi)
            uint4* row = rec.xrow + 5 * q0 + 5 * n;
            row[h] = xb[0];
            row[2 + h] = xb[3];
            // half 1 stores chunk 3 a second time
            row[4 - h] = make_uint4(h ? xb[3].x : xb[4].x, h ? xb[3].y : xb[4].y,
                                    h ? xb[3].z : xb[4].z, h ? xb[3].w : xb[4].w);
        }
        lookup();
        load_records(grp + 2 * stride);
        // A tile's MFMAs run in eight slots; the vector instructions of a slot
        // turn one pair of the tile before (relu, mask, split) into the next
        // layer's B fragments while the matrix core works, and every weight
        // fragment is read two steps ahead of its use.  The scheduling barriers
        // keep the compiler from gathering either kind together again.
        uint32_t mask0[2] = {0u, 0u}, mask1[2] = {0u, 0u};  // words h and h + 2 (q even, odd)
        uint32_t h0[8][3][4];  // layer 1's B fragments [k-step][part][dword]
        uint32_t h1[2][4];     // layer 2's of one k-step
        f32x16 c, d;           // a tile in the making, the one before
        f32x4 lg = {0.f, 0.f, 0.f, 0.f};  // the sample's logits over this lane's features
        const f32x16 zero = {};
        auto pair0 = [&](int T, int j) {  // pair j (rows 2j, 2j + 1 of the lane) of tile T
            uint32_t(*f)[4] = h0[2 * T + (j >> 2)];
            split3(relu(d[2 * j]), relu(d[2 * j + 1]), f[0][j & 3], f[1][j & 3], f[2][j & 3]);
            mask_pair(f[0][j & 3], 2 * (2 * T + (j >> 2)) + (j & 1), mask0[(j >> 1) & 1]);
            pin(f[0][j & 3], f[1][j & 3], f[2][j & 3], mask0[(j >> 1) & 1]);
        };
        uint4 w2f;
        auto pair1 = [&](int T, int j) {
            if ((j & 3) == 1) w2f = w2p[8 * (2 * T + (j >> 2))];
            split2(relu(d[2 * j]), relu(d[2 * j + 1]), h1[0][j & 3], h1[1][j & 3]);
            mask_pair(h1[0][j & 3], 2 * (2 * T + (j >> 2)) + (j & 1), mask1[(j >> 1) & 1]);
            pin(h1[0][j & 3], h1[1][j & 3], mask1[0], mask1[1]);
            if ((j & 3) == 3) {  // layer 2's k-step 2T + j / 4
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    lg = mfma4x4x4(w2f.x, w2f.y, h1[p][0], h1[p][1], lg);
                    lg = mfma4x4x4(w2f.z, w2f.w, h1[p][2], h1[p][3], lg);
                }
            }
        };
        // ---- layer 0: H0^T = relu(W0^T X^T + b0) ----
        uint4 fa = w0ab[0], fb = w023[0];
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            if (T == 3) fetch(0, raw);  // the next group's inputs, from here to layer 1's end
            const uint4 f2 = w042[32 * T];
            c = mfma32x32x16(fa, xb[0], zero);
            if (T > 0) pair0(T - 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            c = mfma32x32x16(fa, xb[1], c);
            if (T > 0) pair0(T - 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            const uint4 f3 = w034[32 * T];
            c = mfma32x32x16(fa, xb[2], c);
            if (T > 0) pair0(T - 1, 2);
            __builtin_amdgcn_sched_barrier(0);
            c = mfma32x32x16(fb, xb[3], c);
            if (T > 0) pair0(T - 1, 3);
            __builtin_amdgcn_sched_barrier(0);
            const uint4 f4 = w04b[32 * T];
            c = mfma32x32x16(fb, xb[6], c);
            if (T > 0) pair0(T - 1, 4);
            __builtin_amdgcn_sched_barrier(0);
            fa = T < 3 ? w0ab[32 * (T + 1)] : w1p[0];
            c = mfma32x32x16(f2, xb[4], c);
            if (T > 0) pair0(T - 1, 5);
            __builtin_amdgcn_sched_barrier(0);
            fb = T < 3 ? w023[32 * (T + 1)] : w1p[64];
            c = mfma32x32x16(f3, xb[5], c);
            if (T > 0) pair0(T - 1, 6);
            __builtin_amdgcn_sched_barrier(0);
            c = mfma32x32x16(f4, xb[7], c);
            if (T > 0) pair0(T - 1, 7);
            __builtin_amdgcn_sched_barrier(0);
            d = c;
        }
        // ---- layer 1: H1^T = relu(W1^T H0^T + b1); layer 2 over its tiles ----
#pragma unroll
        for (int T = 0; T < 4; ++T) {
            uint4 fn = w1p[64 * (9 * T + 2)];
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
            c = mfma32x32x16(fa, sm.ones[h], zero);
            fa = fb;
            fb = fn;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                fn = w1p[64 * min(9 * T + ks + 3, 35)];
                c = mfma32x32x16(fa, frag(h0[ks][0]), c);
                c = mfma32x32x16(fa, frag(h0[ks][1]), c);
                c = mfma32x32x16(fa, frag(h0[ks][2]), c);
                fa = fb;
                fb = fn;
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
        store_x(v);
        wave_lds_fence();
        // ---- the masks and rgb ----
        {
            uint32_t* mw = rec.relu + 8 * q0 + 8 * n + h;
            mw[0] = mask0[0];
            mw[2] = mask0[1];
            mw[4] = mask1[0];
            mw[6] = mask1[1];
            // the two lane halves' sums: half h is left with logit h, both with
            // logit 2; half h finishes channel h, half 0
            // channel 2 too (half 1 writes the unused fourth)
            const auto r01 = __builtin_amdgcn_permlane32_swap(
                __float_as_uint(lg[0]), __float_as_uint(lg[1]), false, false);
            const float x = __uint_as_float(r01[0]) + __uint_as_float(r01[1]);
            const float y = lg[2] + __shfl_xor(lg[2], 32, 64);
            const float a = sigmoidf_(x + b2a), b = sigmoidf_(y + b2b);
            float* rgb = reinterpret_cast<float*>(rec.rgb + q0) + 4 * n + h;
            rgb[0] = alive ? a : 0.f;
            rgb[2] = alive && h == 0 ? b : 0.f;
        }
    }
}

// Backward weights as MFMA A fragments in LDS, [tile][k-step][lane] (each
// wave's W1 rows for the g_H0 product, 32 x 128, sit in its registers):
//   W2  [8 row tiles of 16 hidden][64] x 8 bytes   (K = 16 logits, 3 used)
//   W0  [4 k-steps of 32 hidden][64] x 16 bytes    (rows: the 12 features)
constexpr int kBw2Frags = 8 * 64, kBw0Frags = 4 * 64;

// ---- backward ----------------------------------------------------------------
// One workgroup of 8 wavefronts per CU (two per SIMD); wave w owns hidden
// features [16w, 16w + 16) of both hidden layers, except in the g_H0 product
// (phase 8), where it owns features [32(w/2), +32) of samples [16(w%2), +16).
// Per group of 32 records three stages of work, each pairing products that
// do not depend on one another:
//   A  H0^T = W0^T X^T + b0 under the forward's ReLU mask m0    -> A1h, H0f
//      g_H1^T = W2 g_L^T masked by m1                           -> G1h, G1l, G1f
//   B  H1^T = W1^T H0^T + b1 under the forward's mask m1         -> F2
//      g_H0^T = W1 g_H1^T masked by m0                          -> A2h, A2l, F3
//      dW1 += H0^T g_H1; the next group's records are parked
//   C  dW2 += H1^T g_L; dW0 += X^T g_H0; waves 0-1: g_X^T = W0[0:12] g_H0^T
//      over the whole hidden layer, written from registers as the records'
//      feature gradients
// run as two barrier-separated steps: group k's A with group k-1's C, then
// group k's B.  The input rows X come whole from the forward pass (features,
// encoding, bias input), so group k+1's A needs nothing computed after group
// k's B.
// H0 and H1 are recomputed for the dW operands only (from hi parts, one MFMA
// per product): the masks come from the forward pass (per-record words), so the
// backward applies exactly the ReLU pattern the forward applied.
// X (features, encoding, bias), the per-sample adjoints and the flags are
// double-buffered, so the next group's inputs are staged while this one runs.
constexpr int kBwdWaves = 8;
struct alignas(16) SmemBwd {
    uint4 Bw0[kBw0Frags];
    uint2 Bw2[kBw2Frags];
    uint32_t relu[2][GS * 8];  // the forward's ReLU mask words of each record
    uint16_t Xh[2][GS * XM];
    uint16_t Xf[2][XF_ROWS * FM];
    uint16_t A1h[GS * SM];               // H0 (hi), sample-major
    uint16_t G1h[GS * SM], G1l[GS * SM]; // g_H1, sample-major
    uint16_t A2h[GS * SM], A2l[GS * SM]; // g_H0, sample-major
    uint16_t GLh[2][GS * GM], GLl[2][GS * GM];
    uint16_t H0f[128 * FM];              // H0, feature-major
    uint16_t F2[128 * FM];               // H1, feature-major
    uint16_t G1f[128 * FM];              // g_H1, feature-major
    uint16_t F3[128 * FM];               // g_H0, feature-major
    uint16_t GLf[2][16 * FM];
    float gsig[2][GS];
    uint32_t bits[2][GS];
};

__global__ void __launch_bounds__(64 * kBwdWaves) k_mlp_bwd(StepParams P, MlpPacked W,
                                                            RayBuffers R, Records rec,
                                                            float* __restrict__ dw_partial) {
    constexpr int NTH = 64 * kBwdWaves;
    __shared__ SmemBwd sm;
    const int tid = threadIdx.x;
    const int wv = tid >> 6, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
    const int f0 = 16 * wv;
    const int fr = f0 + 4 * g;  // the 4 features of this lane's D fragment rows
    const int pr = lane < GS / kBwdWaves ? wv * (GS / kBwdWaves) + lane : -1;  // staging lanes

    // forward weight slices in registers (this wave's rows of W0^T and W1^T)
    bf16x8 A0[2], A1[4];
    float b0v[4], b1v[4];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) A0[kt] = ld_frag(W.w0t + (f0 + r16) * 64 + 32 * kt + 8 * g);
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) A1[kt] = ld_frag(W.w1t + (f0 + r16) * 128 + 32 * kt + 8 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        b0v[i] = W.b0[fr + i];
        b1v[i] = W.b1[fr + i];
    }
    // the g_H0 product's tile of this wave: hidden features 32 fb .. +31 (two
    // row tiles) of samples 16 sh .. +15; W1 rows [32 in][128 out] as MFMA A
    // fragments, in registers
    const int fb = wv >> 1, sh = wv & 1;
    bf16x8 Bw1r[2][4];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
            Bw1r[mt][kt] = ld_frag(W.w1 + (32 * fb + 16 * mt + r16) * 128 + 32 * kt + 8 * g);
    // the other backward weights -> LDS
    for (int f = tid; f < kBw2Frags + kBw0Frags; f += NTH) {
        const int ln = f & 63, gg = ln >> 4, rr = ln & 15;
        if (f < kBw2Frags) {  // W2 [128 in][32 out (3 used)], K = 16
            const int t = f >> 6;
            sm.Bw2[f] = *reinterpret_cast<const uint2*>(W.w2 + (16 * t + rr) * 32 + 4 * gg);
        } else {  // W0 rows 0..15 [16][128]
            const int q = f - kBw2Frags, kt = q >> 6;
            sm.Bw0[q] = *reinterpret_cast<const uint4*>(W.w0 + rr * 128 + 32 * kt + 8 * gg);
        }
    }
    f32x4 dW0[3], dW1[8], dW2;
    float db1[4] = {0.f, 0.f, 0.f, 0.f}, db2[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < 3; ++a) dW0[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int a = 0; a < 8; ++a) dW1[a] = f32x4{0.f, 0.f, 0.f, 0.f};
    dW2 = f32x4{0.f, 0.f, 0.f, 0.f};

    // constant parts of the double buffers: X columns 40..63, feature-major X
    // rows 40..47, logits 3..15
    for (int e = tid; e < 2 * GS * 24; e += NTH) {
        const int b = e / (GS * 24), row = (e / 24) % GS, col = 40 + e % 24;
        sm.Xh[b][row * XM + col] = 0;
    }
    for (int e = tid; e < 2 * (XF_ROWS - 40) * FM; e += NTH) {
        const int b = e / ((XF_ROWS - 40) * FM);
        sm.Xf[b][40 * FM + e % ((XF_ROWS - 40) * FM)] = 0;
    }
    for (int e = tid; e < 2 * GS * GM; e += NTH) {
        if (e % GM >= 3) {
            (&sm.GLh[0][0])[e] = 0;
            (&sm.GLl[0][0])[e] = 0;
        }
    }
    for (int e = tid; e < 2 * 16 * FM; e += NTH)
        if ((e % (16 * FM)) >= 3 * FM) (&sm.GLf[0][0])[e] = 0;

    const int64_t total = min((int64_t)R.total[0], P.capacity);
    const int64_t ngroups = (total + GS - 1) / GS;
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    const uint4 zu4 = make_uint4(0u, 0u, 0u, 0u);

    // register prefetch of a group's records: the staging lanes (4 per wave, a
    // record each) take its flags, adjoints and ReLU masks; the row lanes (20
    // per wave) one 16-byte fifth of its input row each.  Every address
    // follows from the record index alone, so the loads of the next group are
    // issued at the start of the current one and land during its products.
    float4 p_adj = z4;
    uint32_t p_bits = 0u;
    uint4 p_r0 = zu4, p_r1 = zu4, p_x = zu4;
    const int xe = (lane >= 32 && lane < 52) ? wv * 20 + (lane - 32) : -1;
    const int xr = xe / 5, xj = xe % 5;  // row lane: record, 8-column part
    auto stage = [&](int64_t grp) {
        const int64_t q = grp * GS + pr;
        p_adj = z4;
        p_bits = 0u;
        p_r0 = p_r1 = zu4;
        if (pr >= 0 && grp < ngroups && q < total) {
            p_bits = __float_as_uint(rec.ab[q].y);
            p_adj = rec.adj[q];
            p_r0 = reinterpret_cast<const uint4*>(rec.relu)[2 * q];  // ReLU masks
            p_r1 = reinterpret_cast<const uint4*>(rec.relu)[2 * q + 1];
        }
        const int64_t qx = grp * GS + xr;
        p_x = zu4;
        if (xe >= 0 && grp < ngroups && qx < total) p_x = rec.xrow[5 * qx + xj];
    };
    // staged records -> buffer b: flags, adjoints (dL/dlogit as (hi, lo) pairs,
    // dL/dsigma), ReLU masks, and the input rows (X columns 0..39, sample-major
    // and feature-major)
    auto park = [&](int b) {
        if (pr >= 0) {
            sm.bits[b][pr] = p_bits;  // zero for records past the end
            sm.gsig[b][pr] = p_adj.w;
            reinterpret_cast<uint4*>(&sm.relu[b][8 * pr])[0] = p_r0;
            reinterpret_cast<uint4*>(&sm.relu[b][8 * pr])[1] = p_r1;
            const float gl[3] = {p_adj.x, p_adj.y, p_adj.z};
            db2[0] += gl[0];
            db2[1] += gl[1];
            db2[2] += gl[2];
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                uint16_t h, l;
                split_bf(gl[o], h, l);
                sm.GLh[b][pr * GM + o] = h;
                sm.GLl[b][pr * GM + o] = l;
                sm.GLf[b][o * FM + pr] = h;
            }
        }
        if (xe >= 0) {
            *reinterpret_cast<uint4*>(&sm.Xh[b][xr * XM + 8 * xj]) = p_x;  // 16-byte aligned
            const uint32_t w4[4] = {p_x.x, p_x.y, p_x.z, p_x.w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                sm.Xf[b][(8 * xj + 2 * c) * FM + xr] = (uint16_t)(w4[c] & 0xffffu);
                sm.Xf[b][(8 * xj + 2 * c + 1) * FM + xr] = (uint16_t)(w4[c] >> 16);
            }
        }
    };
    // stage C of a group whose g_H0 and H1 sit in A2h/A2l, F3 and F2 (its
    // inputs in buffer b, its records from pbase): dW2, dW0 and the records'
    // feature gradients
    auto finish = [&](int b, int64_t pbase) {
        // dW2[in = f0 + row][out] += sum over the group's samples H1[s][in] gL[s][out]
        dW2 = mfma16x16x32(ld_frag(&sm.F2[(f0 + r16) * FM + 8 * g]),
                           ld_frag(&sm.GLf[b][r16 * FM + 8 * g]), dW2);
        {
            const bf16x8 bh = ld_frag(&sm.F3[(f0 + r16) * FM + 8 * g]);
#pragma unroll
            for (int mi = 0; mi < 3; ++mi)
                dW0[mi] = mfma16x16x32(ld_frag(&sm.Xf[b][(16 * mi + r16) * FM + 8 * g]), bh, dW0[mi]);
        }
        if (wv < NT) {
            const int nt = wv;
            f32x4 gx = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) {
                const int go = (16 * nt + r16) * SM + 32 * kt + 8 * g;
                gx = mfma_w(as_bf8(sm.Bw0[kt * 64 + lane]), ld_frag(&sm.A2h[go]),
                            ld_frag(&sm.A2l[go]), gx);
            }
            // lane (g, r16): features 4g..4g+3 of sample 16 nt + r16 = part g of its
            // record's gradient; part 3 carries dL/dsigma
            const int sidx = 16 * nt + r16;
            const int64_t q = pbase + sidx;
            if (q < total) {
                const uint32_t bits = sm.bits[b][sidx];
                float4 v = z4;
                if (g < 3) {
                    if (bits & kAliveW) v = make_float4(gx[0], gx[1], gx[2], gx[3]);
                } else {
                    v.x = sm.gsig[b][sidx];
                }
                rec.grad[4 * q + g] = v;
            }
        }
    };

    stage(blockIdx.x);
    park(0);
    __syncthreads();
    int cb = 0;          // buffer of the current group
    int64_t pbase = -1;  // the previous group, whose stage C is pending (-1: none)

    for (int64_t grp = blockIdx.x; grp < ngroups; grp += gridDim.x) {  // uniform bound
        const int64_t base = grp * GS, next = grp + gridDim.x;
        stage(next);  // in flight during this group's products, parked at its end
        // ---- 1. this group's stage A: H0^T slice = W0^T X^T + b0 under the
        //         forward's mask -> A1h, H0f; g_H1^T slice = W2[slice] g_L^T under
        //         the mask -> G1h, G1l, G1f.  The previous group's stage C ----
        uint32_t m0 = 0u, m1 = 0u;  // the forward's ReLU masks: bit at(nt, i)
        auto at = [](int nt, int i) { return 16 * (i & 1) + 2 * nt + (i >> 1); };
        {
            // features fr..fr+3: bits 2wv, 16 + 2wv, 2wv + 1, 17 + 2wv of word g
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint32_t* mw = &sm.relu[cb][8 * (16 * nt + r16)];
                m0 |= ((mw[g] >> (2 * wv)) & 0x30003u) << (nt * 2);
                m1 |= ((mw[4 + g] >> (2 * wv)) & 0x30003u) << (nt * 2);
            }
        }
        f32x4 acc[NT];  // starting at the bias, as in the forward
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{b0v[0], b0v[1], b0v[2], b0v[3]};
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int xo = (16 * nt + r16) * XM + 32 * kt + 8 * g;
                acc[nt] = mfma16x16x32(A0[kt], ld_frag(&sm.Xh[cb][xo]), acc[nt]);
            }
        }
        {
            const s16x4 a = __builtin_bit_cast(s16x4, sm.Bw2[wv * 64 + lane]);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                f32x4 c4 = {0.f, 0.f, 0.f, 0.f};
                const int go = (16 * nt + r16) * GM + 4 * g;
                c4 = mfma16x16x16(a, ld_frag4(&sm.GLh[cb][go]), c4);
                c4 = mfma16x16x16(a, ld_frag4(&sm.GLl[cb][go]), c4);
                float gv[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    gv[i] = keep_if(m1, at(nt, i), c4[i]);
                    db1[i] += gv[i];
                }
                st_act<true>(sm.G1h, sm.G1l, sm.G1f, 16 * nt + r16, fr, lane, gv);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = keep_if(m0, at(nt, i), acc[nt][i]);
            st_hi_fm(sm.A1h, sm.H0f, 16 * nt + r16, fr, lane, h);
        }
        if (pbase >= 0) finish(cb ^ 1, pbase);
        __syncthreads();
        // ---- 2. B. H1^T slice = W1^T H0^T + b1 under the mask -> F2 (dW2 only);
        //         g_H0^T tile = W1[rows] g_H1^T under the mask -> A2h, A2l, F3;
        //         dW1 += H0^T g_H1; the next group's records are parked ----
        // (g_H0 in 32 features x 16 samples per wave: half the g_H1 reads of 16 x 32)
        f32x4 acc2[2];
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) acc2[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const int go = (16 * sh + r16) * SM + 32 * kt + 8 * g;
            const bf16x8 bh = ld_frag(&sm.G1h[go]), bl = ld_frag(&sm.G1l[go]);
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) acc2[mt] = mfma_w(Bw1r[mt][kt], bh, bl, acc2[mt]);
        }
        {
            // dW1[in][out] += sum over samples H0[s][in] g_H1[s][out]; this wave's
            // block: inputs 64 (wv & 1) .. +63, outputs 32 (wv >> 1) .. +31 (fewer
            // LDS reads than a full column of 128 inputs x 16 outputs)
            const int i0 = 64 * (wv & 1), o0 = 32 * (wv >> 1);
            const bf16x8 b0 = ld_frag(&sm.G1f[(o0 + r16) * FM + 8 * g]);
            const bf16x8 b1 = ld_frag(&sm.G1f[(o0 + 16 + r16) * FM + 8 * g]);
#pragma unroll
            for (int mi = 0; mi < 4; ++mi) {
                const bf16x8 a = ld_frag(&sm.H0f[(i0 + 16 * mi + r16) * FM + 8 * g]);
                dW1[2 * mi] = mfma16x16x32(a, b0, dW1[2 * mi]);
                dW1[2 * mi + 1] = mfma16x16x32(a, b1, dW1[2 * mi + 1]);
            }
        }
        {
            // g_H0 masked by the layer-0 bits of features 32 fb .. +31
            const uint32_t mw = sm.relu[cb][8 * (16 * sh + r16) + g] >> (4 * fb);
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                float gv[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    gv[i] = keep_if(mw, 16 * (i & 1) + 2 * mt + (i >> 1), acc2[mt][i]);
                st_act<true>(sm.A2h, sm.A2l, sm.F3, 16 * sh + r16, 32 * fb + 16 * mt + 4 * g, lane,
                             gv);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = f32x4{b1v[0], b1v[1], b1v[2], b1v[3]};
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const int ho = (16 * nt + r16) * SM + 32 * kt + 8 * g;
                acc[nt] = mfma16x16x32(A1[kt], ld_frag(&sm.A1h[ho]), acc[nt]);
            }
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            float h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = keep_if(m1, at(nt, i), acc[nt][i]);
            st_fm(sm.F2, 16 * nt + r16, fr, lane, h);
        }
        park(cb ^ 1);  // the next group's records, loaded at this group's start
        __syncthreads();
        pbase = base;
        cb ^= 1;
    }
    if (pbase >= 0) finish(cb ^ 1, pbase);  // the loop ended on a barrier

    // ---- flush this workgroup's dW partial ----
    float* out = dw_partial + (int64_t)blockIdx.x * kPartStride;
#pragma unroll
    for (int mi = 0; mi < 3; ++mi)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int in = 16 * mi + 4 * g + i, o = f0 + r16;
            if (in < 39)
                out[kW0 + in * 128 + o] = dW0[mi][i];
            else if (in == 39)
                out[kB0 + o] = dW0[mi][i];
        }
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int in = 64 * (wv & 1) + 16 * (t >> 1) + 4 * g + i;
            const int o = 32 * (wv >> 1) + 16 * (t & 1) + r16;
            out[kW1 + in * 128 + o] = dW1[t][i];
        }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (r16 < 3) out[kW2 + (fr + i) * 3 + r16] = dW2[i];
        float v = db1[i];
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        v += __shfl_xor(v, 8, 64);
        if (r16 == 0) out[kB1 + fr + i] = v;
    }
    // db2 was accumulated by the staging lanes (park); the loop ended on a barrier,
    // so gsig[0] is free for the per-wave sums
#pragma unroll
    for (int o = 0; o < 3; ++o) {
        float v = pr >= 0 ? db2[o] : 0.f;
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        if (lane == 0) sm.gsig[0][4 * wv + o] = v;
    }
    __syncthreads();
    if (tid < 3) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < kBwdWaves; ++w) v += sm.gsig[0][4 * w + tid];
        out[kB2 + tid] = v;
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
