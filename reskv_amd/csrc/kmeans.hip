// Lloyd k-means over pre-RoPE K or V, one independent problem per (batch, head).
//
// Reference loop (reskv/compression.py:37-53): each iteration assigns every
// token to its nearest centre, then replaces each centre by the mean of its
// members.  K (value_mode = 0) keeps an empty cluster's previous centre and
// carries fp32 centres; V (value_mode = 1) sets an empty cluster to zero and
// rounds centres to fp16 after every update.  The returned ids come from the
// last assignment, i.e. against the centres before the final update.
//
// Centre tables (kmeans_prep_kernel, then kmeans_update_kernel every
// iteration): each fp32 centre is split into fp16 hi + lo rows, stored with
// |c|^2, padded to a multiple of 16 rows (padding rows are zero with an
// infinite norm).  They are written once per iteration, so the assignment
// workgroups load ready matrix-core operands instead of rebuilding them.  The
// fp16 norms of the V tokens, which the V rule needs in every iteration, are
// written by the first one.
//
// Assignment (kmeans_assign_kernel): the distance GEMM S^T = C X^T runs on the
// matrix cores (v_mfma_f32_16x16x32f16).  Tokens are fp16 already and
// C X^T = C_hi X^T + C_lo X^T keeps fp32 accuracy (c_hi * x and c_lo * x are
// exact in fp32, sums are fp32).  Each lane holds one token's distances to 4
// centres per 16, so the argmin (lowest index on ties) is a scan in registers
// and two lane swaps across the four lanes sharing the token.  The distance
// follows the rule the reference applies to the tensor:
//   K (compression.py:38, fp32 cdist): |c|^2 - 2 <x, c> in fp32 (|x|^2 is
//     common to a token);
//   V, Lloyd (compression.py:27, 38, fp16 cdist in the mm formulation):
//     fp16(|x|^2_h + |c|^2_h - 2 <x, c>), clamped at zero, square-rooted to
//     fp16; |.|^2_h is the fp16 sum of fp16-rounded squares;
//   V, decode groups (compression.py:61-64):
//     fp16(|x|^2_h + |c|^2_h) - 2 <x, c> in fp32.
// Member sums are a second matrix-core product, onehot(ids)^T X, whose X operand
// comes from the staged token rows through LDS transpose reads.  One-hot entries
// and tokens are exact in fp16 and the products accumulate in fp32, in an order
// that does not depend on the launch; counts are integer LDS adds.  Sums, counts
// and centres are deterministic, and equal for paired and separate runs.
// Update (kmeans_update_kernel): a workgroup adds the partials of four clusters of a
// problem, or of one where there are more than four partials, in a fixed order, and
// writes the new centres and their tables.
#include "common.h"
#include "../../include/reskv_hip.h"
using namespace reskv;

namespace {

typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;

constexpr int kSub = 16;           // tokens per MFMA sub-tile
constexpr int kChunk = 256;        // tokens per chunk of the member sums
constexpr int kCUs = 256;          // compute units of an MI355X
constexpr int kXPitch = kDim + 8;  // halves per staged token row (16-byte aligned rows)
constexpr int kParts = 4;          // interleaved parts of a problem's chunk sums (chunk k belongs to part k % 4)

__device__ __forceinline__ half8_t as_h8(uint4 v) { return __builtin_bit_cast(half8_t, v); }

// (distance, index) minimum with the lower index winning ties
__device__ __forceinline__ void argmin_step(float& d, int& i, float od, int oi) {
    const bool take = od < d || (od == d && oi < i);
    d = take ? od : d;
    i = take ? oi : i;
}

// Tables are kept in matrix-core operand order: the 16 x 32 block (centres
// 16 nb + col, channels 32 q + 8 grp + [0, 8)) that lane 16 grp + col of the
// assignment needs for piece q of centre block nb sits at 16-byte slot
// (4 nb + q) * 64 + 16 grp + col, so each operand load is 1 KB contiguous.
__device__ __forceinline__ int operand_slot_half(int c, int d) {
    return (((c >> 4) * 4 + (d >> 5)) * 64 + ((d >> 3) & 3) * 16 + (c & 15)) * 8 + (d & 7);
}

// Centre c of one problem's tables from the fp32 centre v held by 128 threads
// (channel = thread % 128; s_w: their two floats of LDS).  Every thread of the
// workgroup calls it (it holds a barrier); those without a centre pass active = false.  K rows carry an fp16 lo
// part and the fp32 |c|^2; V rows (fp16 centres) carry the fp16 norm of the
// reference's cdist, the fp16 sum of fp16-rounded squares.
__device__ __forceinline__ void store_tables(float v, bool active, bool pad, bool value, int c,
                                             uint16_t* __restrict__ hi, uint16_t* __restrict__ lo,
                                             float* __restrict__ norm, float* s_w) {
#pragma clang fp contract(off)
    const int t = threadIdx.x & (kDim - 1);
    if (active) {
        const uint16_t hb = f2h(v);
        const int o = operand_slot_half(c, t);
        hi[o] = hb;
        lo[o] = value ? (uint16_t)0 : f2h(v - h2f(hb));
        const float sq = value ? h2f(f2h(v * v)) : v * v;  // V: v is fp16, v*v exact in fp32
        const float w = wave_sum(sq);
        if ((t & 63) == 0) s_w[t >> 6] = w;
    }
    __syncthreads();
    if (active && t == 0) *norm = pad ? INFINITY : (value ? h2f(f2h(s_w[0] + s_w[1])) : s_w[0] + s_w[1]);
}

// Where the problems live: problems [0, split) are rows of tensor 0 and
// [split, BH) rows of tensor 1 (a layer's K and V clustered in one pass);
// problems >= vfrom follow the V rules (fp16 centres, empty -> 0, no lo part).
struct Problems {
    const uint16_t* x[2];  // tokens fp16 [problems, T, 128]
    int32_t* ids[2];       // ids int32 [problems, T]
    uint16_t* out[2];      // final centres fp16 [problems, C, 128]
    int split, vfrom;
};
__device__ __forceinline__ int side_of(const Problems& P, long bh) { return bh >= P.split ? 1 : 0; }

// One workgroup (128 threads) per (padded centre row, problem).
__global__ void __launch_bounds__(kDim) kmeans_prep_kernel(const float* __restrict__ centers, uint16_t* __restrict__ thi,
                                                           uint16_t* __restrict__ tlo, float* __restrict__ tnorm, int C,
                                                           int Cp, int vfrom) {
    __shared__ float s_w[2];
    const int c = blockIdx.x;
    const long bh = blockIdx.y;
    const bool pad = c >= C;
    const float v = pad ? 0.0f : centers[(bh * C + c) * kDim + threadIdx.x];
    const long head = bh * Cp * kDim;
    store_tables(v, true, pad, bh >= vfrom, c, thi + head, tlo + head, tnorm + bh * Cp + c, s_w);
}

// Row indices of the initial centres (at most kMaxClusters), passed by value.
struct InitRows {
    int idx[kMaxClusters];
};

// As kmeans_prep_kernel, with the initial centre c of problem bh taken from
// token idx[c] of that problem's rows (fp16, exact in fp32), also written to
// the fp32 centre array.
__global__ void __launch_bounds__(kDim) kmeans_prep_rows_kernel(Problems P, InitRows ir, float* __restrict__ centers,
                                                                uint16_t* __restrict__ thi, uint16_t* __restrict__ tlo,
                                                                float* __restrict__ tnorm, int T, int C, int Cp) {
    __shared__ float s_w[2];
    const int c = blockIdx.x;
    const long bh = blockIdx.y;
    const bool pad = c >= C;
    const int side = side_of(P, bh);
    const long pb = bh - (side ? P.split : 0);
    float v = 0.0f;
    if (!pad) {
        v = h2f(P.x[side][(pb * T + ir.idx[c]) * kDim + threadIdx.x]);
        centers[(bh * C + c) * kDim + threadIdx.x] = v;
    }
    const long head = bh * Cp * kDim;
    store_tables(v, true, pad, bh >= P.vfrom, c, thi + head, tlo + head, tnorm + bh * Cp + c, s_w);
}

// Four fp16 values, 2.0 where a byte of id4 equals the byte repeated in `mine`
// and 0 elsewhere.  All bytes are below 64: 0x40 - byte keeps bit 6 exactly for a
// zero difference and never borrows from the next byte, and 0x4000 is fp16 2.0.
__device__ __forceinline__ half4_t one_hot4(uint32_t id4, uint32_t mine) {
    const uint32_t e = (0x40404040u - (id4 ^ mine)) & 0x40404040u;
    return __builtin_bit_cast(half4_t, make_uint2(__builtin_amdgcn_perm(0u, e, 0x010C000Cu),
                                                  __builtin_amdgcn_perm(0u, e, 0x030C020Cu)));
}

// |c|^2 of centre r of a lane's four
__device__ __forceinline__ float cnorm(float4 n, int r) { return r == 0 ? n.x : r == 1 ? n.y : r == 2 ? n.z : n.w; }

// (distance, index) minimum over the four lanes holding one token (lanes
// col + 16 g): every lane ends with the token's nearest centre.
__device__ __forceinline__ void token_argmin(float& bd, int& bi) {
    const auto pd = __builtin_amdgcn_permlane32_swap((uint32_t)f2i(bd), (uint32_t)f2i(bd), false, false);
    const auto pi = __builtin_amdgcn_permlane32_swap((uint32_t)bi, (uint32_t)bi, false, false);
    bd = i2f((int)pd[0]);
    bi = (int)pi[0];
    argmin_step(bd, bi, i2f((int)pd[1]), (int)pi[1]);
    const auto qd = __builtin_amdgcn_permlane16_swap((uint32_t)f2i(bd), (uint32_t)f2i(bd), false, false);
    const auto qi = __builtin_amdgcn_permlane16_swap((uint32_t)bi, (uint32_t)bi, false, false);
    bd = i2f((int)qd[0]);
    bi = (int)qi[0];
    argmin_step(bd, bi, i2f((int)qd[1]), (int)qi[1]);
}
__device__ __forceinline__ float token_min(float v) {
    const auto a = __builtin_amdgcn_permlane32_swap((uint32_t)f2i(v), (uint32_t)f2i(v), false, false);
    v = fminf(i2f((int)a[0]), i2f((int)a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap((uint32_t)f2i(v), (uint32_t)f2i(v), false, false);
    return fminf(i2f((int)b[0]), i2f((int)b[1]));
}
__device__ __forceinline__ int token_min_index(int v) {
    const auto a = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
    v = min((int)a[0], (int)a[1]);
    const auto b = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
    return min((int)b[0], (int)b[1]);
}

// fp16 norm of a token as the reference's fp16 cdist forms it: each square
// rounded to fp16, summed in fp32 (this lane's 32 channels, then the four lanes
// of the token; the pairwise sums are commutative, so all four lanes agree),
// rounded to fp16.
__device__ __forceinline__ float token_half_norm(const uint4* xq) {
#pragma clang fp contract(off)
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t w[4] = {xq[q].x, xq[q].y, xq[q].z, xq[q].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float a = h2f((uint16_t)(w[j] & 0xFFFFu)), b = h2f((uint16_t)(w[j] >> 16));
            acc += h2f(f2h(a * a));  // a * a is exact in fp32; one rounding to fp16
            acc += h2f(f2h(b * b));
        }
    }
    const auto p = __builtin_amdgcn_permlane32_swap((uint32_t)f2i(acc), (uint32_t)f2i(acc), false, false);
    acc = i2f((int)p[0]) + i2f((int)p[1]);
    const auto q = __builtin_amdgcn_permlane16_swap((uint32_t)f2i(acc), (uint32_t)f2i(acc), false, false);
    acc = i2f((int)q[0]) + i2f((int)q[1]);
    return h2f(f2h(acc));
}

// For a non-negative fp16 value d (as float): M^2, with M the midpoint between
// the correctly rounded fp16 square root of d and the next fp16 value above
// it.  An fp16 value e has the same fp16 root as d exactly when d <= e < M^2
// (a root is never exactly a midpoint; M has 12 significant bits, so M^2 is
// exact in fp32).  The hardware root is within one fp16 step after rounding
// and is corrected against the midpoints on both sides.
__device__ __forceinline__ float root_bound_sq(float d) {
#pragma clang fp contract(off)
    const uint16_t sb = f2h(__builtin_sqrtf(d));
    float sv = h2f(sb);
    const float up = h2f((uint16_t)(sb + 1)), dn = sb ? h2f((uint16_t)(sb - 1)) : 0.0f;
    const float mhi = 0.5f * (sv + up), mlo = 0.5f * (sv + dn);
    uint16_t rb = sb;
    if (mhi * mhi < d) rb = (uint16_t)(sb + 1);
    else if (sb && mlo * mlo > d) rb = (uint16_t)(sb - 1);
    if (rb >= 0x7C00u) return INFINITY;  // root is infinite: only d itself qualifies
    sv = h2f(rb);
    const float m = 0.5f * (sv + h2f((uint16_t)(rb + 1)));
    return m * m;
}

// Work split of the assignment over a workgroup's waves.  A chunk's 16 sub-tiles
// are summed as r_j = S_{j+4} + S_j, j = 0..3, S_w being sub-tile w, then w + 8; the
// four sub-tiles of an r_j are staged and summed together.  A group of waves works
// on JU of them at a time, one sub-tile per wave; for the member sums its waves
// split the channels in four and, for more than 32 centres, the centre blocks in
// two.  G = 4 groups share a chunk, or one group (G = 1) takes all four r_j in turn.
template <int NB, int G>
struct Split {
    static constexpr int JU = NB <= 2 ? 1 : 2;
    static constexpr int GW = 4 * JU;                 // waves per group
    static constexpr int MB = (NB + JU - 1) / JU;     // centre blocks per wave in the member sums
    static constexpr int NH = 2;                      // 16-channel blocks per wave
    static constexpr int US = 4 * JU;                 // sub-tiles per unit
    static constexpr int waves = GW * G, threads = kWave * waves;
    static constexpr int turns = 4 / (JU * G);        // units of a chunk that a group takes
    static_assert(JU * G * turns == 4 && (G == 1 || JU == 1), "the four r_j of a chunk");
};
// Sub-tile e of r_j (order of summation).
__device__ __forceinline__ int sub_of(int j, int e) { return j + (e < 2 ? 4 : 0) + (e & 1 ? 8 : 0); }

// One workgroup: chunks slot, slot + slots, ... of problem bh (256 tokens each).
//
// Per unit: the wave's sub-tile of token rows goes from its registers to LDS and,
// with the centre operands in LDS, through the distance products; the registers
// then take the next sub-tile's rows, requested before the ids are found, so that
// the loads have the rest of the unit to arrive.  After a barrier the group forms its member
// sums over the unit, each wave for its own channels and centres, so that a sum
// never leaves its lane: no reduction over waves.  The one-hot operand is made from
// four id bytes at a time (2.0 = 0x4000 where a byte equals the lane's cluster; the
// doubled sums are exact and halved at the end).
// Sums are formed in one fixed order whatever slots and G are: r_j as above,
// ((r_0 + r_1) + r_2) + r_3 per chunk, and the chunks of one part (k % 4) in
// increasing order.  A workgroup therefore takes one chunk or a whole part (slots = 4).
//
// thi/tlo fp16 [BH, 16 NB, 128] and tnorm fp32 [BH, 16 NB] are the centre
// tables; psum fp32 [BH, slots, C, 128] and pcnt int [BH, slots, C].  xnorm holds
// the V tokens' fp16 norms [V problems, T]: written when xnorm_new, read otherwise.
// LO: some problem has fp32 centres (V problems skip the lo product).
//
// SUMS: one Lloyd iteration.  Otherwise the ids alone (decode groups): psum, pcnt
// and xnorm are null, the V rule is the groups', and a wave takes its sub-tiles in
// increasing order and ends with the tokens, since a group is a fraction of a chunk
// (8 problems of 64 tokens, C = 33: K 8.2 -> 7.0 us, V 7.5 -> 6.3; 1024 problems, C = 32:
// 25.4 -> 23.6 and 26.4 -> 23.1, with one kernel for both purposes before).
//
// Bound: reading the rows and the VALU work (argmin, one-hot operands) take about
// 0.1 ms each per iteration of 256 problems x 8128 tokens and overlap through four
// independent four-wave workgroups per CU (128 VGPRs, 34 KB of LDS).  The whole
// K-means of that size, 10 iterations: 2330 -> 1556 us (1479 with the update below);
// 16 problems x 8192: 214 -> 182 us; 48 problems x 1999, C = 48, 15 iterations:
// 444 -> 329 us (288).  Two groups of waves per chunk (half the turns) measured
// slower on 512 to 2048 workgroups: 189 against 182 us, 316 against 274.  The kernel
// before had eight waves reduce 16 KB sums each through LDS for every chunk, wrote
// a 16 KB partial per 64 KB of tokens, and (C > 32) fitted one workgroup per CU.
template <int NB, bool LO, int G, bool SUMS>
__global__ void __launch_bounds__((Split<NB, G>::threads)) __attribute__((amdgpu_waves_per_eu(4)))
kmeans_assign_kernel(
    Problems P, const uint16_t* __restrict__ thi, const uint16_t* __restrict__ tlo, const float* __restrict__ tnorm,
    float* __restrict__ psum, int* __restrict__ pcnt, float* __restrict__ xnorm, int xnorm_new, int T, int C,
    int chunks) {
    using W = Split<NB, G>;
    constexpr int CP = NB * 16, MB = W::MB, NH = W::NH, JU = W::JU, US = W::US;
    constexpr int kTab = CP * kDim / 8;                 // 16-byte slots of a centre table
    constexpr int kRows = US * kSub * kXPitch;          // halves of a group's staged rows
    constexpr int kSumPitch = kDim + 4;  // floats: the four rows that a wave writes at once on different banks
    constexpr int kSumBytes = G > 1 ? 4 * CP * kSumPitch * 4 : 0;  // the groups' r_j (reuse the rows)
    constexpr int kRowBytes = G * kRows * 2 > kSumBytes ? G * kRows * 2 : kSumBytes;
    __shared__ __align__(16) uint8_t s_rows[SUMS ? kRowBytes : 16];
    __shared__ __align__(16) uint4 s_hi[kTab];
    __shared__ __align__(16) uint4 s_lo[LO ? kTab : 1];
    __shared__ __align__(16) uint8_t s_id[G * US * kSub];
    __shared__ int s_cnt[CP];
    const int slot = blockIdx.x, slots = gridDim.x;
    const long bh = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave / W::GW, gw = wave % W::GW;  // group, wave of the group
    const int col = lane & 15, grp = lane >> 4;     // MFMA lane coordinates
    const int side = side_of(P, bh);
    const long pb = bh - (side ? P.split : 0);
    const uint16_t* __restrict__ x = P.x[side] + pb * T * kDim;
    int32_t* __restrict__ ids = P.ids[side] + pb * T;
    const bool vrule = bh >= P.vfrom;  // workgroup-uniform
    float* __restrict__ xn_row = SUMS && vrule ? xnorm + (bh - P.vfrom) * T : nullptr;
    uint16_t* s_x = reinterpret_cast<uint16_t*>(s_rows) + g * kRows;
    uint8_t* g_id = s_id + g * US * kSub;

    // token operand: lane (col, grp) holds token t0 + col, channels 32 q + 8 grp +
    // [0, 8) for piece q, so the four lanes of a token read 64 contiguous bytes.
    // Buffer loads past the chunk's tokens return zeros: without a branch around
    // them the registers are not copied (and the loads waited for) at a join.
    uint4 xr[4];
    auto load_sub = [&](int k, int sub) {
        const int left = T - k * kChunk;  // <= 0 past the last chunk
        // uniform values, said so: a descriptor in vector registers would be loaded from lane by lane
        const int rows = __builtin_amdgcn_readfirstlane(left < 0 ? 0 : (left < kChunk ? left : kChunk));
        const uint64_t base = reinterpret_cast<uint64_t>(x + (rows ? (long)k * kChunk * kDim : 0));
        const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)base);
        const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(base >> 32));
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<void*>((uint64_t)hi << 32 | lo), 0, rows * kDim * 2, 0x00020000);
        const int off = (sub * kSub + col) * kDim * 2 + 16 * grp;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            xr[q] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 64 * q, 0, 0));
    };
    // the wave's sub-tile in turn u of a chunk
    auto sub_in = [&](int u) {
        return SUMS ? sub_of((u * G + g) * JU + (gw >> 2), gw & 3) : (u * G + g) * US + gw;
    };
    load_sub(slot, sub_in(0));

    // centre operands: lane (col, grp) reads centre nb*16 + col at the same channels,
    // one contiguous 1 KB wave read per piece (operand-order tables)
    {
        const uint4* ghi = reinterpret_cast<const uint4*>(thi + bh * CP * kDim);
        const uint4* glo = reinterpret_cast<const uint4*>(tlo + bh * CP * kDim);
        for (int i = tid; i < kTab; i += W::threads) {
            s_hi[i] = ghi[i];
            if constexpr (LO)
                if (!vrule) s_lo[i] = glo[i];
        }
        for (int i = tid; i < CP; i += W::threads) s_cnt[i] = 0;
    }
    // |c|^2 of the centres nb*16 + 4*grp + r whose distances this lane holds
    float4 cn[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) cn[nb] = *reinterpret_cast<const float4*>(tnorm + bh * CP + nb * 16 + 4 * grp);
    __syncthreads();

    // twice the part's sums: clusters 16*(nb0 + b) + 4*grp + r, channels d0 + 16*h + col
    float4_t part[MB][NH];
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int h = 0; h < NH; ++h) part[b][h] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
    const int nb0 = MB * (gw >> 2), d0 = 32 * (gw & 3);
    const uint32_t mine0 = (uint32_t)(16 * nb0 + col) * 0x01010101u;
    // transpose reads: lane i of 16-lane row r points at token 4r + i/4, channel
    // d0 + 4*(i%4) and receives tokens 4r + (0..3), channel d0 + i
    const uint16_t* xt = s_x + (4 * grp + (col >> 2)) * kXPitch + d0 + 4 * (col & 3);

    // ids of the wave's sub-tile at t0 (token rows in xr), staged with its rows
    auto assign_sub = [&](int t0, int k_next, int sub_next) {
        const bool live = t0 + col < T;
        if constexpr (SUMS) {
            // rows past T are zeros, so that they add nothing
            uint4* row = reinterpret_cast<uint4*>(s_x + (gw * kSub + col) * kXPitch + 8 * grp);
#pragma unroll
            for (int q = 0; q < 4; ++q) row[4 * q] = xr[q];
        }
        // S^T = C X^T: lane (col, grp) gets <c, x> for token t0 + col and
        // centres nb*16 + 4*grp + r
        float4_t acc[NB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[nb] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
        if (LO && !vrule) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(s_hi[(nb * 4 + q) * 64 + lane]), as_h8(xr[q]), acc[nb], 0, 0, 0);
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(s_lo[LO ? (nb * 4 + q) * 64 + lane : 0]), as_h8(xr[q]), acc[nb], 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as_h8(s_hi[(nb * 4 + q) * 64 + lane]), as_h8(xr[q]), acc[nb], 0, 0, 0);
        }
        float xn = 0.0f;
        if (vrule) {
            if (SUMS && !xnorm_new) {
                xn = xn_row[min(t0 + col, T - 1)];
            } else {
                xn = token_half_norm(xr);
                if (SUMS && grp == 0 && live) xn_row[t0 + col] = xn;
            }
        }
        load_sub(k_next, sub_next);  // the rows are staged and multiplied: their registers take the next ones
        int bi;  // index less 4 * grp within the lane's scan
        if (!vrule) {
            // K: nearest of this lane's centres, scanned in increasing index
            // order (a strict < keeps the lower index on ties), then across the
            // four row groups holding the same token
            float bd = fmaf(-2.0f, acc[0][0], cn[0].x);
            bi = 0;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (nb == 0 && r == 0) continue;
                    const float d = fmaf(-2.0f, acc[nb][r], cnorm(cn[nb], r));
                    const bool take = d < bd;
                    bd = take ? d : bd;
                    bi = take ? nb * 16 + r : bi;
                }
            bi += 4 * grp;
            token_argmin(bd, bi);
        } else {
            if constexpr (!SUMS) {
                // decode groups: fp32(fp16(|x|^2 + |c|^2) - 2 <x, c>), lowest index on
                // ties, which all centres are for a token whose fp16 norm is infinite
                constexpr int kNone = 1 << 20;
                float bd = INFINITY;
                bi = kNone;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float e = h2f(f2h(xn + cnorm(cn[nb], r)));
                        const float d = fmaf(-2.0f, acc[nb][r], e);
                        const bool take = d < bd;
                        bd = take ? d : bd;
                        bi = take ? nb * 16 + r : bi;
                    }
                bi += 4 * grp;
                token_argmin(bd, bi);
                bi = bi >= kNone ? 0 : bi;
            } else {
                // Lloyd: fp16 cdist.  The winner is the lowest index whose fp16
                // root equals the smallest one: with dmin the smallest fp16
                // squared distance and M the midpoint above its fp16 root,
                // that is every d < M^2 (M^2 is exact in fp32), or d == dmin
                // when the root is infinite.
                float d16[NB][4];
                float dmin = INFINITY;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float d = fmaf(-2.0f, acc[nb][r], xn + cnorm(cn[nb], r));
                        d16[nb][r] = fmaxf(h2f(f2h(d)), 0.0f);
                        dmin = fminf(dmin, d16[nb][r]);
                    }
                dmin = token_min(dmin);
                // the largest fp32 value below M^2 (dmin itself when it is infinite)
                const float most = dmin == INFINITY ? dmin : i2f(f2i(root_bound_sq(dmin)) - 1);
                bi = 1 << 20;
#pragma unroll
                for (int nb = NB - 1; nb >= 0; --nb)
#pragma unroll
                    for (int r = 3; r >= 0; --r)
                        if (d16[nb][r] <= most) bi = nb * 16 + r;
                bi = token_min_index(bi + 4 * grp);
            }
        }
        // every lane of column col now holds the id of token t0 + col
        if (grp == 0 && live) ids[t0 + col] = bi;
        if (SUMS && grp == 0) {
            // tokens 4r..4r+3 of all of the unit's sub-tiles are contiguous
            g_id[(col >> 2) * (4 * US) + 4 * gw + (col & 3)] = (uint8_t)(live ? bi & (kMaxClusters - 1) : 0);
            if (live && bi < CP) atomicAdd(&s_cnt[bi], 1);
        }
    };
    // r_j of the unit's jj-th j for this wave's centres and channels
    auto unit_sum = [&](int jj, float4_t (&r)[MB][NH]) {
        const uint4 i4 = *reinterpret_cast<const uint4*>(g_id + grp * (4 * US) + 16 * jj);
        const uint32_t id4[4] = {i4.x, i4.y, i4.z, i4.w};
        float4_t S[2][MB][NH];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int h = 0; h < NH; ++h)
                    if ((e & 1) == 0) S[e >> 1][b][h] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
            half4_t xb[NH];
#pragma unroll
            for (int h = 0; h < NH; ++h)
                xb[h] = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                        (lds_short4_t*)(xt + (4 * jj + e) * kSub * kXPitch + 16 * h)));
#pragma unroll
            for (int b = 0; b < MB; ++b) {
                const half4_t oh = one_hot4(id4[e], mine0 + b * 0x10101010u);
#pragma unroll
                for (int h = 0; h < NH; ++h)
                    S[e >> 1][b][h] = __builtin_amdgcn_mfma_f32_16x16x16f16(oh, xb[h], S[e >> 1][b][h], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                r[b][h] = S[0][b][h] + S[1][b][h];
                asm volatile("" : "+v"(r[b][h]));  // summed here: the S are not held on
            }
    };

    for (int k = slot; k < chunks; k += slots) {
        float4_t tot[MB][NH];
#pragma unroll
        for (int u = 0; u < W::turns; ++u) {
            if (!SUMS && k * kChunk + sub_in(u) * kSub >= T) return;  // uniform over the wave; no barrier follows
            assign_sub(k * kChunk + sub_in(u) * kSub, u + 1 < W::turns ? k : k + slots, sub_in((u + 1) % W::turns));
            // !SUMS, tested at run time in both instances: a chunk's turns in one basic block
            // are slower (16 problems of 8192, 5 iterations 105 us against 96; 64 with C = 64 350 against 264)
            if (psum == nullptr) continue;
            __syncthreads();  // the unit's rows and ids are staged
#pragma unroll
            for (int jj = 0; jj < JU; ++jj) {
                float4_t r[MB][NH];
                unit_sum(jj, r);
                if constexpr (G > 1) {
#pragma unroll
                    for (int b = 0; b < MB; ++b)
#pragma unroll
                        for (int h = 0; h < NH; ++h) tot[b][h] = r[b][h];
                } else {
#pragma unroll
                    for (int b = 0; b < MB; ++b)
#pragma unroll
                        for (int h = 0; h < NH; ++h) tot[b][h] = u == 0 && jj == 0 ? r[b][h] : tot[b][h] + r[b][h];
                }
            }
            __syncthreads();  // the rows are read before the next unit (or the sums) overwrite them
        }
        if constexpr (G == 1) {
            if constexpr (SUMS) {
#pragma unroll
                for (int b = 0; b < MB; ++b)
#pragma unroll
                    for (int h = 0; h < NH; ++h) part[b][h] += tot[b][h];
            }
        } else {
            // one chunk per workgroup: ((r_0 + r_1) + r_2) + r_3, by all threads from LDS
            if constexpr (!SUMS) return;
            float* sums = reinterpret_cast<float*>(s_rows);
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int h = 0; h < NH; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        sums[(g * CP + 16 * (nb0 + b) + 4 * grp + r) * kSumPitch + d0 + 16 * h + col] = tot[b][h][r];
            __syncthreads();
            float4* ps = reinterpret_cast<float4*>(psum + ((bh * slots) + slot) * (long)C * kDim);
            for (int i = tid; i < C * (kDim / 4); i += W::threads) {
                const float* src = sums + (i >> 5) * kSumPitch + 4 * (i & 31);
                float4 v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const float4*>(src + j * CP * kSumPitch);
                // from zero as the parts are, so that a sum of negative zero has their sign
                auto add = [](float a, float b, float c, float d) { return 0.5f * (0.0f + (((a + b) + c) + d)); };
                ps[i] = make_float4(add(v[0].x, v[1].x, v[2].x, v[3].x), add(v[0].y, v[1].y, v[2].y, v[3].y),
                                    add(v[0].z, v[1].z, v[2].z, v[3].z), add(v[0].w, v[1].w, v[2].w, v[3].w));
            }
            for (int i = tid; i < C; i += W::threads) pcnt[(bh * slots + slot) * C + i] = s_cnt[i];
        }
    }
    if (!SUMS || G > 1) return;
    float* ps = psum + ((bh * slots) + slot) * (long)C * kDim + d0 + col;
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = 16 * (nb0 + b) + 4 * grp + r;
            if (c >= C) continue;
#pragma unroll
            for (int h = 0; h < NH; ++h) ps[(long)c * kDim + 16 * h] = 0.5f * part[b][h][r];
        }
    for (int i = tid; i < C; i += W::GW * kWave) pcnt[(bh * slots + slot) * C + i] = s_cnt[i];
}

// The new centres from the partials: per cluster and channel the sums of the four
// parts (chunks of equal residue mod 4, in increasing order), added in order.
// Writes the centre, then either its tables for the next assignment (thi
// non-null) or the fp16 result (thi null).
//
// FEW: at most one partial per part (slots <= 4): 128 threads form a centre from
// four loads and a workgroup takes kParts centres.  Otherwise a workgroup takes one
// centre, 128 threads per part, and the parts meet in LDS.  256 problems with 32
// centres, 4 partials each: 13.5 -> 7 us (8192 workgroups before, 2048 now).
template <bool FEW>
__global__ void __launch_bounds__(kParts * kDim) kmeans_update_kernel(
    Problems P, float* __restrict__ centers, const float* __restrict__ psum, const int* __restrict__ pcnt, int C,
    int Cp, int slots, uint16_t* __restrict__ thi, uint16_t* __restrict__ tlo, float* __restrict__ tnorm) {
    __shared__ float s_part[kParts][kDim];
    __shared__ int s_n[kParts];
    __shared__ float s_w[kParts][2];
    const int d = threadIdx.x & (kDim - 1), quarter = threadIdx.x >> 7;
    const int c = FEW ? blockIdx.x * kParts + quarter : blockIdx.x;
    const long bh = blockIdx.y;
    const bool live = c < C;
    const float* src = psum + (bh * slots) * (long)C * kDim + (live ? c : 0) * kDim + d;
    const int* cnt = pcnt + bh * slots * C + (live ? c : 0);
    float s;
    int n;
    if constexpr (FEW) {
        float p[kParts];
        n = 0;
#pragma unroll
        for (int k = 0; k < kParts; ++k) {
            p[k] = k < slots ? src[(long)k * C * kDim] : 0.0f;
            n += k < slots ? cnt[k * C] : 0;
        }
        s = ((p[0] + p[1]) + p[2]) + p[3];
    } else {
        s = 0.0f;
        n = 0;
#pragma unroll 16
        for (int k = quarter; k < slots; k += kParts) {
            s += src[(long)k * C * kDim];
            n += cnt[k * C];
        }
        s_part[quarter][d] = s;
        if (d == 0) s_n[quarter] = n;
        __syncthreads();
        s = ((s_part[0][d] + s_part[1][d]) + s_part[2][d]) + s_part[3][d];
        n = s_n[0] + s_n[1] + s_n[2] + s_n[3];
    }
    const bool value_mode = bh >= P.vfrom;
    const bool mine = live && (FEW || quarter == 0);
    float nv = 0.0f;
    if (mine) {
        float* cv = centers + (bh * C + c) * kDim + d;
        if (value_mode) {
            nv = n > 0 ? h2f(f2h(s / (float)n)) : 0.0f;  // fp16 centres, empty -> 0
        } else {
            nv = n > 0 ? s / (float)n : *cv;             // fp32 centres, empty keeps
        }
        *cv = nv;
        if (thi == nullptr) {
            const int side = side_of(P, bh);
            P.out[side][((bh - (side ? P.split : 0)) * C + c) * kDim + d] = f2h(nv);
        }
    }
    if (thi == nullptr) return;  // uniform over the workgroup
    const long head = bh * Cp * kDim;
    store_tables(nv, mine, false, value_mode, c, thi + head, tlo + head, tnorm + bh * Cp + c, s_w[FEW ? quarter : 0]);
}

// Workspace: fp32 centres, the fp16 hi/lo tables and norms, chunk partials;
// every array starts on a 256-byte boundary.
struct Layout {
    int Cp, chunks, slots;
    int64_t centers, thi, tlo, tnorm, xnorm, psum, pcnt, total;
};
// Workgroups per problem of the assignment: one per part (each streams its chunks
// and writes one partial) once that fills the chip, else one per chunk.  Up to 32
// centres a part's workgroup has four waves, and two of them per CU are needed (64
// problems of 8192 tokens, 10 iterations: 543 us by parts, 485 by chunks; 128
// problems: 832 against 1025); above 32 it has eight and spares twice the partials
// (C = 64: 32 problems 551 against 447 us, 48 problems 587 against 604, 64
// problems 620 against 765).
int slots_for(int BH, int chunks, int Cp) {
    const int64_t groups = (int64_t)BH * kParts;
    return chunks > kParts && groups >= (Cp <= 32 ? 2 * kCUs : kCUs * 3 / 4) ? kParts : chunks;
}
Layout layout(int BH, int T, int C) {
    Layout L;
    L.Cp = (C + 15) / 16 * 16;
    L.chunks = (T + kChunk - 1) / kChunk;
    L.slots = slots_for(BH, L.chunks, L.Cp);
    int64_t off = 0;
    auto take = [&](int64_t bytes) {
        const int64_t at = off;
        off += (bytes + 255) & ~(int64_t)255;
        return at;
    };
    L.centers = take((int64_t)BH * C * kDim * 4);
    L.thi = take((int64_t)BH * L.Cp * kDim * 2);
    L.tlo = take((int64_t)BH * L.Cp * kDim * 2);
    L.tnorm = take((int64_t)BH * L.Cp * 4);
    L.xnorm = take((int64_t)BH * T * 4);
    L.psum = take((int64_t)BH * L.slots * C * kDim * 4);
    L.pcnt = take((int64_t)BH * L.slots * C * 4);
    L.total = off;
    return L;
}

struct Tables {
    uint16_t* hi;
    uint16_t* lo;
    float* norm;
};

template <int NB, int G>
void launch_nb(bool lo, dim3 grid, hipStream_t st, const Problems& P, const Tables& tb, float* psum, int* pcnt,
               float* xnorm, int xnorm_new, int T, int C, int chunks) {
    const auto kernel = psum != nullptr ? (lo ? kmeans_assign_kernel<NB, true, G, true> : kmeans_assign_kernel<NB, false, G, true>)
                                        : (lo ? kmeans_assign_kernel<NB, true, G, false> : kmeans_assign_kernel<NB, false, G, false>);
    hipLaunchKernelGGL(kernel, grid, dim3(Split<NB, G>::threads), 0, st, P, tb.hi, tb.lo, tb.norm, psum, pcnt, xnorm,
                       xnorm_new, T, C, chunks);
}

int launch_assign(const Problems& P, const Tables& tb, float* psum, int* pcnt, float* xnorm, int xnorm_new, int BH,
                  int T, int C, const Layout& L, hipStream_t st) {
    const dim3 grid(L.slots, BH);
    const bool lo = P.vfrom > 0;
    // a chunk's sub-tiles over 16 waves instead of four turns of four while the
    // grid leaves CUs idle (C = 32, 10 iterations: 64 workgroups 117 against 131 us,
    // 256 134 against 149, 384 192 against 165; with the groups' sums added by all threads
    // since, the first figures are 6 us less)
    const bool wide = L.slots == L.chunks && (int64_t)L.chunks * BH <= kCUs;
    switch (L.Cp / 16) {
    case 1:
        if (wide) launch_nb<1, 4>(lo, grid, st, P, tb, psum, pcnt, xnorm, xnorm_new, T, C, L.chunks);
        else launch_nb<1, 1>(lo, grid, st, P, tb, psum, pcnt, xnorm, xnorm_new, T, C, L.chunks);
        break;
    case 2:
        if (wide) launch_nb<2, 4>(lo, grid, st, P, tb, psum, pcnt, xnorm, xnorm_new, T, C, L.chunks);
        else launch_nb<2, 1>(lo, grid, st, P, tb, psum, pcnt, xnorm, xnorm_new, T, C, L.chunks);
        break;
    case 3: launch_nb<3, 1>(lo, grid, st, P, tb, psum, pcnt, xnorm, xnorm_new, T, C, L.chunks); break;
    default: launch_nb<4, 1>(lo, grid, st, P, tb, psum, pcnt, xnorm, xnorm_new, T, C, L.chunks); break;
    }
    return reskv_host::check_launch("kmeans_assign_kernel");
}

int launch_prep(const float* centers, const Tables& tb, int BH, int C, int Cp, int vfrom, hipStream_t st) {
    hipLaunchKernelGGL(kmeans_prep_kernel, dim3(Cp, BH), dim3(kDim), 0, st, centers, tb.hi, tb.lo, tb.norm, C, Cp,
                       vfrom);
    return reskv_host::check_launch("kmeans_prep_kernel");
}

Tables tables_of(void* workspace, const Layout& L) {
    char* w = (char*)workspace;
    return Tables{(uint16_t*)(w + L.thi), (uint16_t*)(w + L.tlo), (float*)(w + L.tnorm)};
}

int check_pointers(const void* x, const void* workspace) {
    RESKV_REQUIRE(((uintptr_t)x & 15u) == 0, "token rows must be 16-byte aligned");
    RESKV_REQUIRE(((uintptr_t)workspace & 255u) == 0, "k-means workspace must be 256-byte aligned");
    return 0;
}

// torch.linspace(0, T - 1, C).long() (reskv/compression.py:35) as torch
// evaluates it in fp32: step = fl32((T - 1) / (C - 1)); index i < C / 2 is
// fl32(i * step), the others fl32((T - 1) - (C - 1 - i) * step) (one rounding
// of the exact value, as torch's fused form), truncated toward zero.
void linspace_rows(int T, int C, int* idx) {
    if (C == 1) {
        idx[0] = 0;
        return;
    }
    const float end = (float)(T - 1);
    const float step = end / (float)(C - 1);
    for (int i = 0; i < C; ++i) {
        const float v = i < C / 2 ? (float)i * step : fmaf(-(float)(C - 1 - i), step, end);
        idx[i] = (int)v;
    }
}

// Lloyd iterations over BH problems; init[side] holds the initial fp32
// centres of the problems in tensor `side`, or both are null: the tokens at
// linspace(0, T - 1, C) of each problem (T >= C).
int run_kmeans(const Problems& P, const float* const init[2], int BH, int T, int C, int iterations, void* workspace,
               hipStream_t st) {
    const Layout L = layout(BH, T, C);
    const Tables tb = tables_of(workspace, L);
    char* w = (char*)workspace;
    float* centers = (float*)(w + L.centers);
    float* psum = (float*)(w + L.psum);
    int* pcnt = (int*)(w + L.pcnt);
    if (init[0] == nullptr && init[1] == nullptr) {
        InitRows ir{};
        linspace_rows(T, C, ir.idx);
        hipLaunchKernelGGL(kmeans_prep_rows_kernel, dim3(L.Cp, BH), dim3(kDim), 0, st, P, ir, centers, tb.hi, tb.lo,
                           tb.norm, T, C, L.Cp);
        if (reskv_host::check_launch("kmeans_prep_rows_kernel")) return 1;
    } else {
        const size_t row = (size_t)C * kDim * sizeof(float);
        for (int side = 0; side < 2; ++side) {
            const int n = side ? BH - P.split : P.split;
            if (n > 0 && hipMemcpyAsync(centers + (side ? (size_t)P.split * C * kDim : 0), init[side], n * row,
                                        hipMemcpyDeviceToDevice, st) != hipSuccess)
                return reskv_host::check_launch("kmeans centre copy");
        }
        if (launch_prep(centers, tb, BH, C, L.Cp, P.vfrom, st)) return 1;
    }
    float* xnorm = (float*)(w + L.xnorm);
    for (int it = 0; it < iterations; ++it) {
        if (launch_assign(P, tb, psum, pcnt, xnorm, it == 0, BH, T, C, L, st)) return 1;
        const bool last = it == iterations - 1;
        const bool few = L.slots <= kParts;
        const auto update = few ? kmeans_update_kernel<true> : kmeans_update_kernel<false>;
        hipLaunchKernelGGL(update, dim3(few ? (C + kParts - 1) / kParts : C, BH), dim3(kParts * kDim), 0, st, P, centers,
                           psum, pcnt, C, L.Cp, L.slots, last ? nullptr : tb.hi, tb.lo, tb.norm);
        if (reskv_host::check_launch("kmeans_update_kernel")) return 1;
    }
    return 0;
}

}  // namespace

extern "C" int64_t reskv_kmeans_workspace_bytes(int BH, int T, int C) {
    if (BH <= 0 || T <= 0 || C <= 0) return 0;
    return layout(BH, T, C).total;
}

extern "C" int reskv_kmeans_assign(const void* x, const float* centers, int32_t* ids, int BH, int T, int C,
                                   int value_mode, void* workspace, int64_t workspace_bytes, void* stream) {
    RESKV_REQUIRE(x && centers && ids, "null pointer argument");
    RESKV_REQUIRE(BH > 0 && T > 0, "problem sizes must be positive");
    RESKV_REQUIRE(C >= 1 && C <= kMaxClusters, "centroid count must be in [1, 64]");
    RESKV_REQUIRE(value_mode == 0 || value_mode == 1, "value_mode must be 0 (K) or 1 (V)");
    RESKV_REQUIRE(workspace && workspace_bytes >= reskv_kmeans_workspace_bytes(BH, T, C),
                  "k-means workspace too small");
    if (check_pointers(x, workspace)) return 1;
    const Layout L = layout(BH, T, C);
    const Tables tb = tables_of(workspace, L);
    const int vfrom = value_mode ? 0 : BH;
    const Problems P{{(const uint16_t*)x, (const uint16_t*)x}, {ids, ids}, {nullptr, nullptr}, BH, vfrom};
    hipStream_t st = (hipStream_t)stream;
    if (launch_prep(centers, tb, BH, C, L.Cp, vfrom, st)) return 1;
    return launch_assign(P, tb, nullptr, nullptr, nullptr, 0, BH, T, C, L, st);
}

extern "C" int reskv_linspace_rows(int T, int C, int32_t* rows) {
    RESKV_REQUIRE(rows != nullptr, "null pointer argument");
    RESKV_REQUIRE(C >= 1 && C <= kMaxClusters && T >= C, "need 1 <= C <= 64 and T >= C");
    int idx[kMaxClusters];
    linspace_rows(T, C, idx);
    for (int i = 0; i < C; ++i) rows[i] = idx[i];
    return 0;
}

extern "C" int reskv_kmeans(const void* x, const float* centers_init, void* centers_out, int32_t* ids,
                            int BH, int T, int C, int iterations, int value_mode, void* workspace,
                            int64_t workspace_bytes, void* stream) {
    RESKV_REQUIRE(x && centers_out && ids, "null pointer argument");
    RESKV_REQUIRE(centers_init || T >= C, "linspace initial centres need T >= C");
    RESKV_REQUIRE(BH > 0 && T > 0, "problem sizes must be positive");
    RESKV_REQUIRE(C >= 1 && C <= kMaxClusters, "centroid count must be in [1, 64]");
    RESKV_REQUIRE(iterations >= 1, "iterations must be positive");
    RESKV_REQUIRE(workspace && workspace_bytes >= reskv_kmeans_workspace_bytes(BH, T, C),
                  "k-means workspace too small");
    if (check_pointers(x, workspace)) return 1;
    const uint16_t* xh = (const uint16_t*)x;
    uint16_t* out = (uint16_t*)centers_out;
    const Problems P{{xh, xh}, {ids, ids}, {out, out}, BH, value_mode ? 0 : BH};
    const float* const init[2] = {centers_init, centers_init};
    return run_kmeans(P, init, BH, T, C, iterations, workspace, (hipStream_t)stream);
}

extern "C" int reskv_kmeans_kv(const void* k, const void* v, const float* init_k, const float* init_v, void* out_k,
                               void* out_v, int32_t* ids_k, int32_t* ids_v, int BH, int T, int C, int iterations,
                               void* workspace, int64_t workspace_bytes, void* stream) {
    RESKV_REQUIRE(k && v && out_k && out_v && ids_k && ids_v, "null pointer argument");
    RESKV_REQUIRE((init_k == nullptr) == (init_v == nullptr), "give both initial centre arrays or neither");
    RESKV_REQUIRE(init_k || T >= C, "linspace initial centres need T >= C");
    RESKV_REQUIRE(BH > 0 && T > 0, "problem sizes must be positive");
    RESKV_REQUIRE(C >= 1 && C <= kMaxClusters, "centroid count must be in [1, 64]");
    RESKV_REQUIRE(iterations >= 1, "iterations must be positive");
    RESKV_REQUIRE(workspace && workspace_bytes >= reskv_kmeans_workspace_bytes(2 * BH, T, C),
                  "k-means workspace too small");
    if (check_pointers(k, workspace) || check_pointers(v, workspace)) return 1;
    const Problems P{{(const uint16_t*)k, (const uint16_t*)v}, {ids_k, ids_v}, {(uint16_t*)out_k, (uint16_t*)out_v},
                     BH, BH};
    const float* const init[2] = {init_k, init_v};
    return run_kmeans(P, init, 2 * BH, T, C, iterations, workspace, (hipStream_t)stream);
}
