// Residual encoders: four lanes per token (eight for 4:16).  Few rows, rows of a few
// tokens and inputs that are not 16-byte aligned take one wavefront per token, lane L
// owning channels L and L+64.
//
// Every encoder computes r = f32(x) - f32(c[id]) and ranks channels by the
// 15-bit magnitude of fp16(r) with ties going to the lower channel index
// (reskv/csrc/compression.cu:80-118, 184-203, 287-313; reskv/compression.py:75-89).
// In the one-wavefront kernels the rank key is made unique by appending the
// inverted channel index, so "top-k" is a single threshold on that composite key:
//   ckey(d) = (|fp16(r_d)| bits) << 7 | (127 - d).
// Top-k over all 128 channels uses a 22-step bitwise threshold search on
// wave ballots; top-k inside a 16-channel tile counts larger keys from LDS.
#include "common.h"

using namespace reskv;

namespace {

constexpr int kWavesPerBlock = 4;

// The tensors one launch encodes: side 0 and, for a layer's K and V in one
// launch, side 1 (grid dimension y for the 4:16 encoder, z for the bitmap
// encoder selects the side).
struct EncSides {
    const uint16_t* x[2];     // tokens fp16 [B*H*T, 128]
    const uint16_t* cent[2];  // centroids fp16 [B*H, C, 128]
    const int32_t* ids[2];    // cluster ids [B*H*T]
    uint16_t* payload[2];
    void* meta[2];
    int C[2];
};

struct Residual {
    float r0, r1;     // channels L, L+64
    uint32_t m0, m1;  // |fp16(r)| as 15-bit integers (order == value order)
};

__device__ __forceinline__ Residual load_residual(const uint16_t* __restrict__ keys,
                                                  const uint16_t* __restrict__ cent,
                                                  const int32_t* __restrict__ ids,
                                                  long row, long bh, int C, int lane) {
    int cid = ids[row];
    cid = cid < 0 ? 0 : (cid > C - 1 ? C - 1 : cid);  // compression.cu:83-84
    const uint16_t* x = keys + row * kDim;
    const uint16_t* c = cent + (bh * C + cid) * kDim;
    Residual r;
    r.r0 = h2f(x[lane]) - h2f(c[lane]);
    r.r1 = h2f(x[lane + kHalf]) - h2f(c[lane + kHalf]);
    r.m0 = f2h(r.r0) & 0x7FFFu;
    r.m1 = f2h(r.r1) & 0x7FFFu;
    return r;
}

__device__ __forceinline__ uint32_t ckey(uint32_t mag, int d) { return (mag << 7) | (uint32_t)(127 - d); }

// Threshold tau with exactly k composite keys >= tau (keys are unique).
__device__ __forceinline__ uint32_t topk_threshold(uint32_t k0, uint32_t k1, int k) {
    uint32_t prefix = 0;
#pragma unroll
    for (int bit = 21; bit >= 0; --bit) {
        const uint32_t cand = prefix | (1u << bit);
        const int cnt = __builtin_popcountll(ballot(k0 >= cand)) + __builtin_popcountll(ballot(k1 >= cand));
        prefix = cnt >= k ? cand : prefix;
    }
    return prefix;
}

// Number of keys in the lane's 16-channel tile that outrank its own key.
__device__ __forceinline__ int tile_rank(const uint32_t* tile_keys, uint32_t mine) {
    int rank = 0;
#pragma unroll
    for (int j = 0; j < 16; ++j) rank += tile_keys[j] > mine ? 1 : 0;
    return rank;
}

__device__ __forceinline__ uint64_t bitrev64(uint64_t v) {
    return ((uint64_t)__builtin_bitreverse32((uint32_t)v) << 32) | __builtin_bitreverse32((uint32_t)(v >> 32));
}

__global__ void __launch_bounds__(256) encode_qtile_kernel(
    const uint16_t* __restrict__ keys, const uint16_t* __restrict__ cent,
    const int32_t* __restrict__ ids, uint16_t* __restrict__ payload, int32_t* __restrict__ meta,
    long rows, int T, int C, int nnz, int struct_index) {
    __shared__ uint32_t s_keys[kWavesPerBlock][kDim];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int per_tile = nnz >> 3;
    for (long row = (long)blockIdx.x * kWavesPerBlock + wave; row < rows;
         row += (long)gridDim.x * kWavesPerBlock) {
        const long bh = row / T;
        const Residual r = load_residual(keys, cent, ids, row, bh, C, lane);
        const uint32_t k0 = ckey(r.m0, lane), k1 = ckey(r.m1, lane + kHalf);
        s_keys[wave][lane] = k0;
        s_keys[wave][lane + kHalf] = k1;
        wave_sync();
        const int tile0 = lane >> 4, bit = lane & 15;
        const bool sel0 = tile_rank(&s_keys[wave][tile0 * 16], k0) < per_tile;
        const bool sel1 = tile_rank(&s_keys[wave][(tile0 + 4) * 16], k1) < per_tile;
        const uint64_t b0 = ballot(sel0), b1 = ballot(sel1);
        const uint32_t below = (1u << bit) - 1u;
        const uint32_t t0 = (uint32_t)(b0 >> (16 * tile0)) & 0xFFFFu;
        const uint32_t t1 = (uint32_t)(b1 >> (16 * tile0)) & 0xFFFFu;
        uint16_t* prow = payload + row * nnz;
        if (sel0) prow[tile0 * per_tile + __builtin_popcount(t0 & below)] = f2h(r.r0);
        if (sel1) prow[(tile0 + 4) * per_tile + __builtin_popcount(t1 & below)] = f2h(r.r1);
        if (lane < 4) {
            // word w = code(tile 2w) | code(tile 2w+1) << 16
            uint32_t word = 0;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int tile = 2 * lane + half;
                const uint64_t b = tile < 4 ? b0 : b1;
                const uint32_t mask = (uint32_t)(b >> (16 * (tile & 3))) & 0xFFFFu;
                uint32_t code = mask;
                if (struct_index) {
                    code = 0;
                    int rank = 0;
                    for (int i = 0; i < 16; ++i)
                        if ((mask >> i) & 1u) code |= (uint32_t)i << (4 * rank++);
                }
                word |= code << (16 * half);
            }
            meta[row * 4 + lane] = (int32_t)word;
        }
        wave_sync();
    }
}

// ---------------------------------------------------------------------------
// 4 of 16 per tile (structured 4:16 at 75%): eight lanes per token, lane
// 8 t + j owns 16-channel tile j of token t, so a wave encodes 8 tokens and
// every load and store is a contiguous run of the token's row.
//
// fp16(f32(x) - f32(c)) equals the correctly rounded fp16 difference for every
// pair of finite fp16 values (checked exhaustively), so residuals come from
// packed fp16 subtraction.  Each channel j of the tile gets the unique key
//   (|h| << 5) | ((15 - j) << 1) | sign(h)
// (magnitude first, lower channel on ties, the fp16 bits recoverable from the
// key); a selection network yields the top 4 keys, which are then put in
// channel order.
// ---------------------------------------------------------------------------
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef short short2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void cx_desc(uint32_t& a, uint32_t& b) {  // a >= b afterwards
    const uint32_t hi = max(a, b), lo = min(a, b);
    a = hi;
    b = lo;
}
__device__ __forceinline__ void sort4_desc(uint32_t& a, uint32_t& b, uint32_t& c, uint32_t& d) {
    cx_desc(a, b);
    cx_desc(c, d);
    cx_desc(a, c);
    cx_desc(b, d);
    cx_desc(b, c);
}
// a, b: descending lists of 4.  a becomes the descending top 4 of both:
// max(a_i, b_{3-i}) is that set as a bitonic sequence, then a half-cleaner
// merge sorts it.
__device__ __forceinline__ void merge_top4(uint32_t* a, const uint32_t* b) {
    uint32_t c0 = max(a[0], b[3]), c1 = max(a[1], b[2]), c2 = max(a[2], b[1]), c3 = max(a[3], b[0]);
    cx_desc(c0, c2);
    cx_desc(c1, c3);
    cx_desc(c0, c1);
    cx_desc(c2, c3);
    a[0] = c0;
    a[1] = c1;
    a[2] = c2;
    a[3] = c3;
}

__global__ void __launch_bounds__(256) encode_tile4_kernel(EncSides S, long rows, int T, int struct_index) {
    const int side = blockIdx.y;
    const uint16_t* __restrict__ keys = S.x[side];
    const uint16_t* __restrict__ cent = S.cent[side];
    const int32_t* __restrict__ ids = S.ids[side];
    uint16_t* __restrict__ payload = S.payload[side];
    int32_t* __restrict__ meta = static_cast<int32_t*>(S.meta[side]);
    const int C = S.C[side];
    const int lane = threadIdx.x & 63;
    const long row = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * 8 + (lane >> 3);
    const int tile = lane & 7;
    if (row >= rows) return;
    const long bh = row / T;
    int cid = ids[row];
    cid = cid < 0 ? 0 : (cid > C - 1 ? C - 1 : cid);  // compression.cu:83-84
    const uint4* xp = reinterpret_cast<const uint4*>(keys + row * kDim + tile * 16);
    const uint4* cp = reinterpret_cast<const uint4*>(cent + (bh * C + cid) * kDim + tile * 16);
    const uint4 xa = xp[0], xb = xp[1], ca = cp[0], cb = cp[1];
    const uint32_t xw[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
    const uint32_t cw[8] = {ca.x, ca.y, ca.z, ca.w, cb.x, cb.y, cb.z, cb.w};
    uint32_t k[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, xw[i]) - __builtin_bit_cast(half2_t, cw[i]));
        const uint32_t lo = h & 0xFFFFu, hi = h >> 16;
        k[2 * i] = ((lo & 0x7FFFu) << 5) | ((uint32_t)(15 - 2 * i) << 1) | (lo >> 15);
        k[2 * i + 1] = ((hi & 0x7FFFu) << 5) | ((uint32_t)(14 - 2 * i) << 1) | (hi >> 15);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) sort4_desc(k[4 * g], k[4 * g + 1], k[4 * g + 2], k[4 * g + 3]);
    merge_top4(k, k + 4);
    merge_top4(k + 8, k + 12);
    // the top 4 of all 16 (unordered), re-keyed by channel: (15 - j) << 16 | fp16 bits
    uint32_t s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t t = max(k[i], k[11 - i]);
        s[i] = ((t & 0x1Eu) << 15) | ((t & 1u) << 15) | (t >> 5);
    }
    sort4_desc(s[0], s[1], s[2], s[3]);  // ascending channel
    uint2 pw;
    pw.x = (s[0] & 0xFFFFu) | (s[1] << 16);
    pw.y = (s[2] & 0xFFFFu) | (s[3] << 16);
    *reinterpret_cast<uint2*>(payload + row * 32 + tile * 4) = pw;
    uint32_t code = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t j = 15u - (s[i] >> 16);
        code |= struct_index ? j << (4 * i) : 1u << j;
    }
    // word w = code(tile 2w) | code(tile 2w+1) << 16
    const uint32_t other = dpp_u<0xB1>(code);  // quad xor 1: the neighbouring tile
    if ((tile & 1) == 0) meta[row * 4 + (tile >> 1)] = (int32_t)(code | (other << 16));
}

__global__ void __launch_bounds__(256) encode_bitmap_kernel(
    const uint16_t* __restrict__ keys, const uint16_t* __restrict__ cent,
    const int32_t* __restrict__ ids, uint16_t* __restrict__ payload, int64_t* __restrict__ meta,
    long rows, int T, int C, int nnz) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (long row = (long)blockIdx.x * kWavesPerBlock + wave; row < rows;
         row += (long)gridDim.x * kWavesPerBlock) {
        const long bh = row / T;
        const Residual r = load_residual(keys, cent, ids, row, bh, C, lane);
        const uint32_t k0 = ckey(r.m0, lane), k1 = ckey(r.m1, lane + kHalf);
        const uint32_t tau = topk_threshold(k0, k1, nnz);
        const bool sel0 = k0 >= tau, sel1 = k1 >= tau;
        const uint64_t b0 = ballot(sel0), b1 = ballot(sel1);
        uint16_t* prow = payload + row * nnz;
        if (sel0) prow[lanes_below(b0)] = f2h(r.r0);
        if (sel1) prow[__builtin_popcountll(b0) + lanes_below(b1)] = f2h(r.r1);
        // channel d -> bit (63 - d % 64) of word d / 64 (compression.py:87-88)
        if (lane < 2) meta[row * 2 + lane] = (int64_t)bitrev64(lane == 0 ? b0 : b1);
    }
}

// ---------------------------------------------------------------------------
// Selection on bit planes, four lanes per token (lane 4 t + q owns channels
// 32 q .. 32 q + 31 of token t; a wave encodes 16 tokens).
//
// A lane's 32 fp16 residuals are transposed into bit planes: plane b holds bit
// b of every magnitude, bit j of the plane being channel 32 q + j.  The k-th
// largest magnitude is then found from the top plane down with one AND and one
// popcount per plane for all 32 channels: `alive` are the channels that agree
// with the threshold on the planes seen so far, and of these the ones with the
// next bit set are either enough to hold the k-th largest (they stay alive) or
// all above the threshold (they are kept, and the rest stays alive).  What is
// alive after the last plane equals the threshold; ties go to the lower
// channel.  The kept channels come out as a 32-bit mask, which is the metadata
// word of the tile format and the reversed half word of the bitmaps.
//
// Bound: VALU issue.  The transpose takes 16 + 16 byte permutes and 96
// shift / bit-select operations, the 15 planes about 12 instructions each,
// against 224 byte-difference sums and about 260 instructions of sums, flags
// and masks for the byte-plane search this replaced.
// ---------------------------------------------------------------------------
constexpr int kTokensPerWave = 16;
constexpr int kTokensPerBlock = kWavesPerBlock * kTokensPerWave;
constexpr int kRowPadHalves = 8;  // halves after each LDS payload row: 16-byte aligned rows that start on different banks
constexpr int kRowHalves = kTokensPerWave * (kDim + kRowPadHalves);  // LDS halves of a wave's rows, before the dump slots

// Sum over the four lanes of the lane's token (one DPP quad), in every one of them.
__device__ __forceinline__ int quad_sum(int v) {
    v += (int)dpp_u<0xB1>((uint32_t)v);  // quad xor 1
    v += (int)dpp_u<0x4E>((uint32_t)v);  // quad xor 2
    return v;
}
__device__ __forceinline__ float quad_max(float v) {
    v = fmaxf(v, dpp<0xB1>(v));
    return fmaxf(v, dpp<0x4E>(v));
}
// Exclusive prefix sum over the quad, in lane (channel) order.
__device__ __forceinline__ int quad_prefix(int v, int q) {
    int s = v;
    const int a = (int)dpp_u<0x90>((uint32_t)s);  // quad_perm [0,0,1,2]: lane q - 1
    s += q >= 1 ? a : 0;
    const int b = (int)dpp_u<0x44>((uint32_t)s);  // quad_perm [0,1,0,1]: lane q - 2
    s += q >= 2 ? b : 0;
    return s - v;
}

// The lane's 32 channels: tokens and centroid rows as loaded, residuals as fp16 pairs.
struct Lane32 {
    uint32_t x[16], c[16], h[16];  // channels 32 q + 2 i, + 1
};
__device__ __forceinline__ void load_lane32(const uint16_t* __restrict__ keys, const uint16_t* __restrict__ cent,
                                            const int32_t* __restrict__ ids, long row, long bh, int C, int q,
                                            Lane32& L) {
    int cid = ids[row];
    cid = cid < 0 ? 0 : (cid > C - 1 ? C - 1 : cid);  // compression.cu:83-84
    const uint4* xp = reinterpret_cast<const uint4*>(keys + row * kDim + q * 32);
    const uint4* cp = reinterpret_cast<const uint4*>(cent + (bh * C + cid) * kDim + q * 32);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint4 xv = xp[j], cv = cp[j];
        const uint32_t xw[4] = {xv.x, xv.y, xv.z, xv.w}, cw[4] = {cv.x, cv.y, cv.z, cv.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            L.x[4 * j + k] = xw[k];
            L.c[4 * j + k] = cw[k];
            L.h[4 * j + k] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, xw[k]) - __builtin_bit_cast(half2_t, cw[k]));
        }
    }
}

__device__ __forceinline__ uint32_t bit_select(uint32_t m, uint32_t a, uint32_t b) { return (a & m) | (b & ~m); }

// pl[b] = bit b of every channel's fp16 residual (bit j: channel j), b = 0..15.
// Channels j and j + 16 share a dword, so the two 16 x 16 bit matrices in the
// low and high halves are transposed together, in four exchange stages.
__device__ __forceinline__ void bit_planes(const uint32_t* h, uint32_t* pl) {
#pragma unroll
    for (int j = 0; j < 16; ++j)
        pl[j] = __builtin_amdgcn_perm(h[8 + (j >> 1)], h[j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t a = pl[j], b = pl[j + 8];
        pl[j] = __builtin_amdgcn_perm(b, a, 0x06020400u);
        pl[j + 8] = __builtin_amdgcn_perm(b, a, 0x07030501u);
    }
#pragma unroll
    for (int stage = 0; stage < 3; ++stage) {
        const int s = 4 >> stage;
        const uint32_t m = s == 4 ? 0x0F0F0F0Fu : (s == 2 ? 0x33333333u : 0x55555555u);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if (j & s) continue;
            const uint32_t a = pl[j], b = pl[j + s];
            pl[j] = bit_select(m, a, b << s);
            pl[j + s] = bit_select(m, a >> s, b);
        }
    }
}

// Kept channels of the lane.  above: strictly larger than the threshold
// magnitude; kept: those and the lowest-indexed ones equal to it.
struct Kept {
    uint32_t kept, above;
};
// Drops the highest-indexed of the equal channels until `quota` of them are left.
__device__ __forceinline__ uint32_t lowest_bits(uint32_t eq, int quota) {
    for (int n = __builtin_popcount(eq); n > quota; --n) eq &= ~(0x80000000u >> __builtin_clz(eq));
    return eq;
}
// Top nnz of the token's 128 channels (1 <= nnz <= 128).
__device__ __forceinline__ Kept select_token(const uint32_t* pl, int nnz, int q) {
    uint32_t alive = 0xFFFFFFFFu, above = 0;
    int need = nnz;
#pragma unroll
    for (int b = 14; b >= 0; --b) {
        const uint32_t m = alive & pl[b];
        const int n = quad_sum(__builtin_popcount(m));
        const bool enough = n >= need;
        above |= enough ? 0u : m;
        alive = enough ? m : alive ^ m;
        need = enough ? need : need - n;
    }
    int quota = need - quad_prefix(__builtin_popcount(alive), q);
    quota = quota < 0 ? 0 : quota;
    return Kept{above | lowest_bits(alive, quota), above};
}
// Top `per_tile` of each of the lane's two 16-channel tiles (the mask's halves).
__device__ __forceinline__ uint32_t select_tiles(const uint32_t* pl, int per_tile) {
    uint32_t alive = 0xFFFFFFFFu, above = 0;
    int need0 = per_tile, need1 = per_tile;
#pragma unroll
    for (int b = 14; b >= 0; --b) {
        const uint32_t m = alive & pl[b];
        const int n0 = __builtin_popcount(m & 0xFFFFu), n1 = __builtin_popcount(m >> 16);
        const bool e0 = n0 >= need0, e1 = n1 >= need1;
        const uint32_t enough = (e0 ? 0xFFFFu : 0u) | (e1 ? 0xFFFF0000u : 0u);
        above |= m & ~enough;
        alive = bit_select(enough, m, alive ^ m);
        need0 = e0 ? need0 : need0 - n0;
        need1 = e1 ? need1 : need1 - n1;
    }
    return above | lowest_bits(alive & 0xFFFFu, need0) | lowest_bits(alive & 0xFFFF0000u, need1);
}

// Sparse FP16 formats.  TILE: top nnz / 8 of every 16-channel tile with
// LSB-first tile masks; otherwise top nnz of the token with MSB-first bitmaps.
// NNZ: the payload width when it is one of the common ones, else 0 (runtime).
// The kept residuals go to the token's row in the wave's LDS in channel order
// (the others to a dump slot of the lane, so the loop has no branch), and from
// there to the payload as 16-byte stores.
// 8 heads x 8192 tokens, K and V in one launch: 50% bitmap 18.7 -> 15.6 us, 75%
// 17.9 -> 13.9 us (byte planes before), 50% tiles 41.2 -> 16.2 us (one wave per
// token before).  64 heads x 16384 tokens: 231 -> 193, 210 -> 169 and 503 ->
// 208 us, i.e. 4.4, 4.2 and 4.1 TB/s (a large copy reaches 4.9).
template <bool TILE, int NNZ>
__global__ void __launch_bounds__(256) encode_planes_kernel(EncSides S, int T, int nnz_arg, int bh0) {
    __shared__ __align__(16) uint16_t s_rows[kWavesPerBlock][kRowHalves + kWave];
    const int nnz = NNZ ? NNZ : nnz_arg;
    const int side = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane & 3;
    const int t_wave = blockIdx.x * kTokensPerBlock + wave * kTokensPerWave;
    if (t_wave >= T) return;  // whole waves
    const int t = t_wave + (lane >> 2);
    const bool valid = t < T;  // lanes past T compute on the last token and store nothing
    const long bh = (long)bh0 + blockIdx.y;
    const long row = bh * T + (valid ? t : T - 1);
    Lane32 L;
    load_lane32(S.x[side], S.cent[side], S.ids[side], row, bh, S.C[side], q, L);
    uint32_t pl[16];
    bit_planes(L.h, pl);
    const uint32_t sel = TILE ? select_tiles(pl, nnz >> 3) : select_token(pl, nnz, q).kept;
    if constexpr (TILE) {
        // word w = mask(tile 2w) | mask(tile 2w + 1) << 16
        if (valid) static_cast<int32_t*>(S.meta[side])[row * 4 + q] = (int32_t)sel;
    } else {
        // channel d -> bit (63 - d % 64) of word d / 64 (compression.py:87-88):
        // lane 2w holds the high half of word w, lane 2w + 1 the low half
        const uint32_t rev = __builtin_bitreverse32(sel);
        const uint32_t rev_next = dpp_u<0xB1>(rev);
        if (valid && (q & 1) == 0)
            static_cast<int64_t*>(S.meta[side])[row * 2 + (q >> 1)] = (int64_t)(((uint64_t)rev << 32) | rev_next);
    }
    const int kept = __builtin_popcount(sel);
    const int first = TILE ? q * (nnz >> 2) : quad_prefix(kept, q);
    const int pitch = nnz + kRowPadHalves;
    uint16_t* srow = s_rows[wave];
    uint8_t* sbytes = reinterpret_cast<uint8_t*>(srow);
    const uint32_t dump = 2 * (kRowHalves + lane);
    int at = 2 * ((lane >> 2) * pitch + first + kept);  // byte offset past the lane's last kept value
#pragma unroll
    for (int i = 31; i >= 0; --i) {
        const int m = __builtin_amdgcn_sbfe((int)sel, i, 1);  // -1 when channel i is kept
        at += m * 2;
        uint8_t* dst = sbytes + bit_select((uint32_t)m, (uint32_t)at, dump);
        *reinterpret_cast<uint16_t*>(dst) = (uint16_t)(L.h[i >> 1] >> (16 * (i & 1)));
    }
    wave_sync();
    const int ntok = T - t_wave < kTokensPerWave ? T - t_wave : kTokensPerWave;
    uint16_t* grow = S.payload[side] + (bh * T + t_wave) * (long)nnz;  // the wave's rows are contiguous
    if ((nnz & 7) == 0) {
        const int per = nnz >> 3;
        uint4* dst = reinterpret_cast<uint4*>(grow);
        for (int c = lane; c < ntok * per; c += kWave) {
            const int r = c / per;
            dst[c] = *reinterpret_cast<const uint4*>(srow + r * pitch + 8 * (c - r * per));
        }
    } else {
        for (int c = lane; c < ntok * nnz; c += kWave) {
            const int r = c / nnz;
            grow[c] = srow[r * pitch + c - r * nnz];
        }
    }
}

// ---------------------------------------------------------------------------
// Unstructured top-nnz with INT4 / INT2 codes (compression.cu:245-383), on the
// same planes.  With s the fp16-rounded scale, a code is
// clamp(rint(fl32(r / s)), -QMAX, QMAX).  It is formed without a division per
// channel, exactly:
//   INT2: rint(fl32(r / s)) is 0 exactly when |r| <= s / 2.  (s / 2 and the
//   other rounding boundaries b s, b = k + 1/2 <= 7.5, have at most 15
//   significant bits, so they are exact in fp32; if r is not b s, r / s differs
//   from b by at least ulp(b) / m with m the significand of s, 1 <= m < 2, so
//   that fl32(r / s) is not b either.)
//   INT4: t = r * rcp(s) plus one Newton correction is within 2^-20 ulp of r / s
//   before its last rounding, while the quotients nearest a boundary are at
//   least 0.0002 ulp away from rounding to it: rint gives the same integer.
//   Adding 1.5 * 2^23 rounds to the nearest even integer in the low bits, and
//   eight codes biased by 8 are gathered by shift-adds.
// Waves in which a residual is infinite or NaN, a scale is zero or infinite,
// or every kept magnitude ties (the largest |r| in fp32 may then be among the
// dropped channels) take the plain form: the masked maximum, and a division
// per channel.
// K and V of 64 heads x 16384 tokens at 50%: INT4 681 -> 172 us (4.0 TB/s), INT2
// 728 -> 148 us (4.2 TB/s), against the one-wave-per-token kernels, which take
// four lanes' ballots for each of 22 search steps and divide for every channel.
// ---------------------------------------------------------------------------
template <int BITS>
__global__ void __launch_bounds__(256) encode_quant_kernel(const uint16_t* __restrict__ keys,
                                                           const uint16_t* __restrict__ cent,
                                                           const int32_t* __restrict__ ids,
                                                           uint32_t* __restrict__ qtiles,
                                                           uint16_t* __restrict__ qscale, int T, int C, int nnz,
                                                           int bh0) {
#pragma clang fp contract(off)
    constexpr int kQmax = (1 << (BITS - 1)) - 1;
    constexpr int kPerWord = 32 / BITS;
    constexpr int kLaneWords = BITS;  // 32 channels of BITS bits
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane & 3;
    const int t_wave = blockIdx.x * kTokensPerBlock + wave * kTokensPerWave;
    if (t_wave >= T) return;  // whole waves
    const int t = t_wave + (lane >> 2);
    const bool valid = t < T;  // lanes past T compute on the last token and store nothing
    const long bh = (long)bh0 + blockIdx.y;
    const long row = bh * T + (valid ? t : T - 1);
    Lane32 L;
    load_lane32(keys, cent, ids, row, bh, C, q, L);
    uint32_t pl[16];
    bit_planes(L.h, pl);
    const Kept K = select_token(pl, nnz, q);
    const uint32_t sel = K.kept;
    float r[32];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const uint32_t sh = 16u * (i & 1);
        r[i] = h2f((uint16_t)(L.x[i >> 1] >> sh)) - h2f((uint16_t)(L.c[i >> 1] >> sh));
        amax = fmaxf(amax, fabsf(r[i]));
    }
    amax = quad_max(amax);
    // fp16(amax / QMAX) with an IEEE fp32 division, fp16(1) for an all-zero residual
    uint16_t hs = amax > 0.0f ? f2h(amax / (float)kQmax) : f2h(1.0f);
    const uint32_t nonfinite = pl[14] & pl[13] & pl[12] & pl[11] & pl[10];
    const int above = quad_sum(__builtin_popcount(K.above));
    const bool plain = nonfinite != 0 || above == 0 || (hs & 0x7FFFu) == 0 || hs >= 0x7C00u;
    uint32_t w[kLaneWords];
    if (ballot(plain) == 0) {
        const float sf = h2f(hs);
        if constexpr (BITS == 2) {
            const float half_step = 0.5f * sf;
            uint32_t nz = 0, neg = 0;  // bit i: channel i has a nonzero code / is negative
#pragma unroll
            for (int i = 31; i >= 0; --i) {
                nz = __builtin_amdgcn_alignbit(nz, (uint32_t)f2i(half_step - fabsf(r[i])), 31);
                neg = __builtin_amdgcn_alignbit(neg, (uint32_t)f2i(r[i]), 31);
            }
            nz &= sel;
            neg &= nz;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                uint32_t a = (nz >> (16 * k)) & 0xFFFFu, n = (neg >> (16 * k)) & 0xFFFFu;
#pragma unroll
                for (int stage = 0; stage < 4; ++stage) {  // bit i to bit 2 i
                    const int s = 8 >> stage;
                    const uint32_t m = s == 8 ? 0x00FF00FFu : (s == 4 ? 0x0F0F0F0Fu : (s == 2 ? 0x33333333u : 0x55555555u));
                    a = (a | (a << s)) & m;
                    n = (n | (n << s)) & m;
                }
                w[k] = a | (n << 1);  // 01: +1, 11: -1
            }
        } else {
            const float inv = __builtin_amdgcn_rcpf(sf);
            constexpr float kMagic = 12582912.0f;  // 1.5 * 2^23, bits 0x4B400000
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t acc = 0;
#pragma unroll
                for (int j = 7; j >= 0; --j) {
                    const float v = r[8 * k + j];
                    float d = v * inv;
                    d = __builtin_fmaf(__builtin_fmaf(-d, sf, v), inv, d);
                    d = __builtin_amdgcn_fmed3f(d, -7.0f, 7.0f);
                    acc = (acc << 4) + (uint32_t)f2i(d + kMagic);
                }
                acc = (acc - 0x4B400000u * 0x11111111u + 0x88888888u) ^ 0x88888888u;
                // the kept channels' nibbles
                uint32_t m = (sel >> (8 * k)) & 0xFFu;
                m = (m | (m << 12)) & 0x000F000Fu;
                m = (m | (m << 6)) & 0x03030303u;
                m = (m | (m << 3)) & 0x11111111u;
                w[k] = acc & ((m << 4) - m);
            }
        }
    } else {
        amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 32; ++i) amax = fmaxf(amax, (sel >> i) & 1u ? fabsf(r[i]) : 0.0f);
        amax = quad_max(amax);
        hs = amax > 0.0f ? f2h(amax / (float)kQmax) : f2h(1.0f);
        const float sf = h2f(hs);
#pragma unroll
        for (int k = 0; k < kLaneWords; ++k) {
            uint32_t acc = 0;
#pragma unroll
            for (int j = 0; j < kPerWord; ++j) {
                int code = (int)rintf(r[kPerWord * k + j] / sf);
                code = code < -kQmax ? -kQmax : (code > kQmax ? kQmax : code);
                if ((sel >> (kPerWord * k + j)) & 1u) acc |= (uint32_t)(code & ((1 << BITS) - 1)) << (BITS * j);
            }
            w[k] = acc;
        }
    }
    if (!valid) return;
    uint32_t* dst = qtiles + row * (4 * kLaneWords) + kLaneWords * q;
    if constexpr (BITS == 4) *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
    else *reinterpret_cast<uint2*>(dst) = make_uint2(w[0], w[1]);
    if (q == 0) qscale[row] = hs;
}

// ---------------------------------------------------------------------------
// Structured INT4 (compression.cu:153-239): 1 of every 4 channels, four lanes
// per token as above (lane q: subgroups 8 q .. 8 q + 7, i.e. payload word q and
// half a metadata word), so every load and store is a contiguous run.  K and V
// of 64 heads x 16384 tokens: 541 -> 128 us, 4.7 TB/s (a large copy reaches 4.9).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) encode_sint4_kernel(const uint16_t* __restrict__ keys,
                                                           const uint16_t* __restrict__ cent,
                                                           const int32_t* __restrict__ ids,
                                                           int32_t* __restrict__ qpacked, int32_t* __restrict__ qmeta,
                                                           uint16_t* __restrict__ qscale, int T, int C, int bh0) {
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int q = lane & 3;
    const int t_wave = blockIdx.x * kTokensPerBlock + wave * kTokensPerWave;
    if (t_wave >= T) return;  // whole waves
    const int t = t_wave + (lane >> 2);
    const bool valid = t < T;  // lanes past T compute on the last token and store nothing
    const long bh = (long)bh0 + blockIdx.y;
    const long row = bh * T + (valid ? t : T - 1);
    Lane32 L;
    load_lane32(keys, cent, ids, row, bh, C, q, L);
    float v[8];
    uint32_t pos_bits = 0;
    float amax = 0.0f;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        // largest |fp16(r)| of the four, the lower channel on ties: magnitude
        // above the inverted position
        const uint32_t a = L.h[2 * g], b = L.h[2 * g + 1];
        const uint32_t k0 = ((a & 0x7FFFu) << 2) | 3u, k1 = ((a >> 14) & 0x1FFFCu) | 2u;
        const uint32_t k2 = ((b & 0x7FFFu) << 2) | 1u, k3 = (b >> 14) & 0x1FFFCu;
        const uint32_t pos = 3u - (max(max(k0, k1), max(k2, k3)) & 3u);
        const uint32_t xw = pos & 2u ? L.x[2 * g + 1] : L.x[2 * g], cw = pos & 2u ? L.c[2 * g + 1] : L.c[2 * g];
        const uint32_t sh = (pos & 1u) * 16u;
        v[g] = h2f((uint16_t)(xw >> sh)) - h2f((uint16_t)(cw >> sh));
        amax = fmaxf(amax, fabsf(v[g]));
        pos_bits |= pos << (2 * g);
    }
    amax = quad_max(amax);
    const float s = amax > 0.0f ? amax * (1.0f / 7.0f) : 1.0f;  // compression.cu:224
    uint32_t word = 0;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        int code = (int)rintf(v[g] / s);
        code = code < -7 ? -7 : (code > 7 ? 7 : code);
        word |= (uint32_t)(code & 0xF) << (4 * g);
    }
    const uint32_t pos_next = dpp_u<0xB1>(pos_bits);  // quad xor 1: the other half of the metadata word
    if (!valid) return;
    qpacked[row * 4 + q] = (int32_t)word;
    if ((q & 1) == 0) qmeta[row * 2 + (q >> 1)] = (int32_t)(pos_bits | (pos_next << 16));
    if (q == 0) qscale[row] = f2h(s);
}

template <int BITS>
__global__ void __launch_bounds__(256) encode_multibit_kernel(
    const uint16_t* __restrict__ keys, const uint16_t* __restrict__ cent,
    const int32_t* __restrict__ ids, int32_t* __restrict__ qtiles, uint16_t* __restrict__ qscale,
    long rows, int T, int C, int nnz) {
    constexpr int kPerWord = 32 / BITS;
    constexpr int kQmax = (1 << (BITS - 1)) - 1;
    constexpr int kWords = kDim / kPerWord;
    __shared__ uint8_t s_code[kWavesPerBlock][kDim];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (long row = (long)blockIdx.x * kWavesPerBlock + wave; row < rows;
         row += (long)gridDim.x * kWavesPerBlock) {
        const long bh = row / T;
        const Residual r = load_residual(keys, cent, ids, row, bh, C, lane);
        const uint32_t k0 = ckey(r.m0, lane), k1 = ckey(r.m1, lane + kHalf);
        const uint32_t tau = topk_threshold(k0, k1, nnz);
        const bool sel0 = k0 >= tau, sel1 = k1 >= tau;
        const float amax = wave_max(fmaxf(sel0 ? fabsf(r.r0) : 0.0f, sel1 ? fabsf(r.r1) : 0.0f));
        // fp16(amax / QMAX) with an IEEE fp32 division, fp16(1) for an all-zero residual
        const uint16_t hs = amax > 0.0f ? f2h(amax / (float)kQmax) : f2h(1.0f);
        const float sf = h2f(hs);
        int q0 = (int)rintf(r.r0 / sf), q1 = (int)rintf(r.r1 / sf);
        q0 = q0 < -kQmax ? -kQmax : (q0 > kQmax ? kQmax : q0);
        q1 = q1 < -kQmax ? -kQmax : (q1 > kQmax ? kQmax : q1);
        s_code[wave][lane] = sel0 ? (uint8_t)(q0 & ((1 << BITS) - 1)) : 0;
        s_code[wave][lane + kHalf] = sel1 ? (uint8_t)(q1 & ((1 << BITS) - 1)) : 0;
        wave_sync();
        if (lane < kWords) {
            uint32_t word = 0;
#pragma unroll
            for (int i = 0; i < kPerWord; ++i) word |= (uint32_t)s_code[wave][lane * kPerWord + i] << (i * BITS);
            qtiles[row * kWords + lane] = (int32_t)word;
        }
        if (lane == 0) qscale[row] = hs;
        wave_sync();
    }
}

__global__ void __launch_bounds__(256) encode_struct_int4_kernel(
    const uint16_t* __restrict__ keys, const uint16_t* __restrict__ cent,
    const int32_t* __restrict__ ids, int32_t* __restrict__ qpacked, int32_t* __restrict__ qmeta,
    uint16_t* __restrict__ qscale, long rows, int T, int C) {
    __shared__ uint8_t s_nib[kWavesPerBlock][32];
    __shared__ uint8_t s_sel[kWavesPerBlock][32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (long row = (long)blockIdx.x * kWavesPerBlock + wave; row < rows;
         row += (long)gridDim.x * kWavesPerBlock) {
        const long bh = row / T;
        const Residual r = load_residual(keys, cent, ids, row, bh, C, lane);
        // 1 of 4 per subgroup: largest magnitude, lower channel on ties
        const uint32_t sub = (uint32_t)(lane & 3);
        uint32_t c0 = (r.m0 << 2) | (3u - sub), c1 = (r.m1 << 2) | (3u - sub);
        uint32_t x0 = c0, x1 = c1;
        x0 = max(x0, dpp_u<0xB1>(x0));
        x0 = max(x0, dpp_u<0x4E>(x0));
        x1 = max(x1, dpp_u<0xB1>(x1));
        x1 = max(x1, dpp_u<0x4E>(x1));
        const bool sel0 = c0 == x0, sel1 = c1 == x1;
        float v0 = sel0 ? r.r0 : 0.0f, v1 = sel1 ? r.r1 : 0.0f;
        v0 += dpp<0xB1>(v0);
        v0 += dpp<0x4E>(v0);
        v1 += dpp<0xB1>(v1);
        v1 += dpp<0x4E>(v1);
        const float amax = wave_max(fmaxf(fabsf(v0), fabsf(v1)));
        const float s = amax > 0.0f ? amax * (1.0f / 7.0f) : 1.0f;  // compression.cu:224
        int q0 = (int)rintf(v0 / s), q1 = (int)rintf(v1 / s);
        q0 = q0 < -7 ? -7 : (q0 > 7 ? 7 : q0);
        q1 = q1 < -7 ? -7 : (q1 > 7 ? 7 : q1);
        const int g0 = lane >> 2, g1 = g0 + 16;  // subgroup indices of channels L, L+64
        if (sel0) {
            s_nib[wave][g0] = (uint8_t)(q0 & 0xF);
            s_sel[wave][g0] = (uint8_t)sub;
        }
        if (sel1) {
            s_nib[wave][g1] = (uint8_t)(q1 & 0xF);
            s_sel[wave][g1] = (uint8_t)sub;
        }
        wave_sync();
        if (lane < 4) {
            uint32_t word = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) word |= (uint32_t)s_nib[wave][lane * 8 + i] << (4 * i);
            qpacked[row * 4 + lane] = (int32_t)word;
        } else if (lane < 6) {
            const int w = lane - 4;
            uint32_t word = 0;
#pragma unroll
            for (int i = 0; i < 16; ++i) word |= (uint32_t)s_sel[wave][w * 16 + i] << (2 * i);
            qmeta[row * 2 + w] = (int32_t)word;
        } else if (lane == 6) {
            qscale[row] = f2h(s);
        }
        wave_sync();
    }
}

int grid_for(long rows) {
    long blocks = (rows + kWavesPerBlock - 1) / kWavesPerBlock;
    const long cap = 256L * 64;  // enough resident waves to saturate HBM; loop the rest
    return (int)(blocks < cap ? (blocks < 1 ? 1 : blocks) : cap);
}

int check_common(const void* keys, const void* cent, const void* ids, int B, int H, int T, int C) {
    RESKV_REQUIRE(keys && cent && ids, "null input pointer");
    RESKV_REQUIRE(B > 0 && H > 0 && T > 0, "batch, head and token dimensions must be positive");
    RESKV_REQUIRE(C >= 1 && C <= kMaxClusters, "centroid count must be in [1, 64]");
    return 0;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// 4:16 fast path: nnz 32, 16-byte aligned tokens and centroids, 8-byte aligned payload.
bool tile4_ok(const EncSides& S, int sides, int nnz) {
    bool ok = nnz == 32;
    for (int i = 0; i < sides; ++i)
        ok = ok && aligned16(S.x[i]) && aligned16(S.cent[i]) && ((uintptr_t)S.payload[i] & 7u) == 0;
    return ok;
}
int launch_tile4(const EncSides& S, int sides, int B, int H, int T, int struct_index, hipStream_t st) {
    const long rows = (long)B * H * T;
    hipLaunchKernelGGL(encode_tile4_kernel, dim3((int)((rows + 31) / 32), sides), dim3(256), 0, st, S, rows, T,
                       struct_index);
    return reskv_host::check_launch("encode_tile4_kernel");
}

// four-lanes-per-token encoders: 16-byte aligned tokens, centroids and payload.
bool planes_ok(const EncSides& S, int sides) {
    bool ok = true;
    for (int i = 0; i < sides; ++i) ok = ok && aligned16(S.x[i]) && aligned16(S.cent[i]) && aligned16(S.payload[i]);
    return ok;
}
// Whether one wave per token is the faster form of a single-tensor call: its waves do less
// work one after the other, and four lanes per token leave lanes idle where a (batch,
// head) row has few tokens.
//   few: the rows (of 64 tokens) up to which it is, because a wave's latency is all there
//     is.  2048 rows: INT4 3.8 against 4.4 us, INT2 3.9 / 4.2, structured INT4 3.6 / 3.6, and
//     at 4096 4.5 / 4.4, 4.5 / 4.2, 4.0 / 3.6; tiles 3.8 / 4.7 and bitmaps 4.1 / 4.7 at
//     4096 rows, 4.8 / 4.8 and 5.4 / 4.8 at 8192.
//   most: the tokens of a row from which it is not.  65536 rows of one token: INT4 27
//     against 85 us, structured INT4 22 / 50, tiles 20 / 108, bitmaps 25 / 98; four lanes
//     per token take the same for up to 16 tokens, one wave each that many times as long.
bool one_wave_each(long rows, int T, long few, int most) { return rows <= few || T < most; }
constexpr long kFewRows16 = 4096, kFewRowsCodes = 2048;
constexpr int kTokensTiles = 8, kTokensBitmap = 4, kTokensQuant = 4, kTokensSInt4 = 3;

// Calls launch(grid, first (batch, head) row) over all rows: grid y covers at most 65535 of them.
template <typename Launch>
int over_rows(int BH, int T, int sides, const char* what, Launch launch) {
    for (int bh0 = 0; bh0 < BH; bh0 += 65535) {
        launch(dim3((T + kTokensPerBlock - 1) / kTokensPerBlock, BH - bh0 < 65535 ? BH - bh0 : 65535, sides), bh0);
        if (reskv_host::check_launch(what)) return 1;
    }
    return 0;
}
template <bool TILE>
int launch_planes(const EncSides& S, int sides, int B, int H, int T, int nnz, hipStream_t st) {
    return over_rows(B * H, T, sides, "encode_planes_kernel", [&](dim3 grid, int bh0) {
        if (nnz == 64)
            hipLaunchKernelGGL((encode_planes_kernel<TILE, 64>), grid, dim3(256), 0, st, S, T, nnz, bh0);
        else if (nnz == 32)
            hipLaunchKernelGGL((encode_planes_kernel<TILE, 32>), grid, dim3(256), 0, st, S, T, nnz, bh0);
        else
            hipLaunchKernelGGL((encode_planes_kernel<TILE, 0>), grid, dim3(256), 0, st, S, T, nnz, bh0);
    });
}

}  // namespace

extern "C" int reskv_compress_fp16(const void* keys, const void* centroids, const int32_t* ids,
                                   void* payload, int32_t* meta, int B, int H, int T, int C,
                                   int nnz, int struct_index, void* stream) {
    if (check_common(keys, centroids, ids, B, H, T, C)) return 1;
    RESKV_REQUIRE(payload && meta, "null output pointer");
    RESKV_REQUIRE(nnz > 0 && nnz < kDim && nnz % 8 == 0,
                  "FP16 tile encoder requires nnz divisible by 8 and < 128");
    RESKV_REQUIRE(!struct_index || nnz == 32, "4:16 index codes require nnz == 32");
    const long rows = (long)B * H * T;
    const EncSides S{{(const uint16_t*)keys, nullptr}, {(const uint16_t*)centroids, nullptr}, {ids, nullptr},
                     {(uint16_t*)payload, nullptr}, {meta, nullptr}, {C, 0}};
    if (tile4_ok(S, 1, nnz)) return launch_tile4(S, 1, B, H, T, struct_index, (hipStream_t)stream);
    if (planes_ok(S, 1) && !one_wave_each(rows, T, kFewRows16, kTokensTiles))
        return launch_planes<true>(S, 1, B, H, T, nnz, (hipStream_t)stream);
    hipLaunchKernelGGL(encode_qtile_kernel, dim3(grid_for(rows)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)keys, (const uint16_t*)centroids, ids, (uint16_t*)payload, meta,
                       rows, T, C, nnz, struct_index);
    return reskv_host::check_launch("encode_qtile_kernel");
}

extern "C" int reskv_compress_bitmap(const void* keys, const void* centroids, const int32_t* ids,
                                     void* payload, int64_t* meta, int B, int H, int T, int C,
                                     int nnz, void* stream) {
    if (check_common(keys, centroids, ids, B, H, T, C)) return 1;
    RESKV_REQUIRE(payload && meta, "null output pointer");
    RESKV_REQUIRE(nnz > 0 && nnz <= kDim, "nnz must be in [1, 128]");
    const long rows = (long)B * H * T;
    const EncSides S{{(const uint16_t*)keys, nullptr}, {(const uint16_t*)centroids, nullptr}, {ids, nullptr},
                     {(uint16_t*)payload, nullptr}, {meta, nullptr}, {C, 0}};
    if (planes_ok(S, 1) && !one_wave_each(rows, T, kFewRows16, kTokensBitmap))
        return launch_planes<false>(S, 1, B, H, T, nnz, (hipStream_t)stream);
    hipLaunchKernelGGL(encode_bitmap_kernel, dim3(grid_for(rows)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)keys, (const uint16_t*)centroids, ids, (uint16_t*)payload, meta,
                       rows, T, C, nnz);
    return reskv_host::check_launch("encode_bitmap_kernel");
}

extern "C" int reskv_compress_quantized(const void* keys, const void* centroids, const int32_t* ids,
                                        int32_t* qtiles, void* qscale, int B, int H, int T, int C,
                                        int nnz, int bits, void* stream) {
    if (check_common(keys, centroids, ids, B, H, T, C)) return 1;
    RESKV_REQUIRE(qtiles && qscale, "null output pointer");
    RESKV_REQUIRE(nnz == 32 || nnz == 64, "quantised encoder requires nnz in {32, 64}");
    RESKV_REQUIRE(bits == 2 || bits == 4, "quantised encoder requires bits in {2, 4}");
    const long rows = (long)B * H * T;
    // rows read and written with 16-byte (INT2: 8-byte) accesses where they are aligned to them
    if (aligned16(keys) && aligned16(centroids) && aligned16(qtiles) &&
        !one_wave_each(rows, T, kFewRowsCodes, kTokensQuant))
        return over_rows(B * H, T, 1, "encode_quant_kernel", [&](dim3 grid, int bh0) {
            auto kernel = bits == 4 ? encode_quant_kernel<4> : encode_quant_kernel<2>;
            hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)keys,
                               (const uint16_t*)centroids, ids, (uint32_t*)qtiles, (uint16_t*)qscale, T, C, nnz, bh0);
        });
    if (bits == 4)
        hipLaunchKernelGGL(encode_multibit_kernel<4>, dim3(grid_for(rows)), dim3(256), 0, (hipStream_t)stream,
                           (const uint16_t*)keys, (const uint16_t*)centroids, ids, qtiles,
                           (uint16_t*)qscale, rows, T, C, nnz);
    else
        hipLaunchKernelGGL(encode_multibit_kernel<2>, dim3(grid_for(rows)), dim3(256), 0, (hipStream_t)stream,
                           (const uint16_t*)keys, (const uint16_t*)centroids, ids, qtiles,
                           (uint16_t*)qscale, rows, T, C, nnz);
    return reskv_host::check_launch("encode_multibit_kernel");
}

extern "C" int reskv_compress_structured_int4(const void* keys, const void* centroids,
                                              const int32_t* ids, int32_t* qpacked, int32_t* qmeta,
                                              void* qscale, int B, int H, int T, int C, void* stream) {
    if (check_common(keys, centroids, ids, B, H, T, C)) return 1;
    RESKV_REQUIRE(qpacked && qmeta && qscale, "null output pointer");
    const long rows = (long)B * H * T;
    if (aligned16(keys) && aligned16(centroids) && !one_wave_each(rows, T, kFewRowsCodes, kTokensSInt4))
        return over_rows(B * H, T, 1, "encode_sint4_kernel", [&](dim3 grid, int bh0) {
            hipLaunchKernelGGL(encode_sint4_kernel, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t*)keys,
                               (const uint16_t*)centroids, ids, qpacked, qmeta, (uint16_t*)qscale, T, C, bh0);
        });
    hipLaunchKernelGGL(encode_struct_int4_kernel, dim3(grid_for(rows)), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)keys, (const uint16_t*)centroids, ids, qpacked, qmeta,
                       (uint16_t*)qscale, rows, T, C);
    return reskv_host::check_launch("encode_struct_int4_kernel");
}

// A layer's K and V in one launch (grid side dimension); each result equals
// the single-tensor call's.  Inputs that miss the fast path's alignment run
// as two single-tensor calls, and so do many rows of a few tokens (few rows do not:
// 4096 of them take 4.7 us in one launch of four lanes per token, 6.5 in two).
extern "C" int reskv_compress_fp16_kv(const void* k, const void* v, const void* k_centroids,
                                      const void* v_centroids, const int32_t* k_ids, const int32_t* v_ids,
                                      void* k_payload, void* v_payload, int32_t* k_meta, int32_t* v_meta, int B,
                                      int H, int T, int Ck, int Cv, int nnz, int struct_index, void* stream) {
    if (check_common(k, k_centroids, k_ids, B, H, T, Ck) || check_common(v, v_centroids, v_ids, B, H, T, Cv))
        return 1;
    RESKV_REQUIRE(k_payload && v_payload && k_meta && v_meta, "null output pointer");
    const long rows = (long)B * H * T;
    const EncSides S{{(const uint16_t*)k, (const uint16_t*)v}, {(const uint16_t*)k_centroids, (const uint16_t*)v_centroids},
                     {k_ids, v_ids}, {(uint16_t*)k_payload, (uint16_t*)v_payload}, {k_meta, v_meta}, {Ck, Cv}};
    if (tile4_ok(S, 2, nnz) && (!struct_index || nnz == 32))
        return launch_tile4(S, 2, B, H, T, struct_index, (hipStream_t)stream);
    if (planes_ok(S, 2) && !struct_index && nnz > 0 && nnz < kDim && nnz % 8 == 0 &&
        (rows <= kFewRows16 || T >= kTokensTiles))
        return launch_planes<true>(S, 2, B, H, T, nnz, (hipStream_t)stream);
    if (reskv_compress_fp16(k, k_centroids, k_ids, k_payload, k_meta, B, H, T, Ck, nnz, struct_index, stream))
        return 1;
    return reskv_compress_fp16(v, v_centroids, v_ids, v_payload, v_meta, B, H, T, Cv, nnz, struct_index, stream);
}

extern "C" int reskv_compress_bitmap_kv(const void* k, const void* v, const void* k_centroids,
                                        const void* v_centroids, const int32_t* k_ids, const int32_t* v_ids,
                                        void* k_payload, void* v_payload, int64_t* k_meta, int64_t* v_meta, int B,
                                        int H, int T, int Ck, int Cv, int nnz, void* stream) {
    if (check_common(k, k_centroids, k_ids, B, H, T, Ck) || check_common(v, v_centroids, v_ids, B, H, T, Cv))
        return 1;
    RESKV_REQUIRE(k_payload && v_payload && k_meta && v_meta, "null output pointer");
    const long rows = (long)B * H * T;
    RESKV_REQUIRE(nnz > 0 && nnz <= kDim, "nnz must be in [1, 128]");
    const EncSides S{{(const uint16_t*)k, (const uint16_t*)v}, {(const uint16_t*)k_centroids, (const uint16_t*)v_centroids},
                     {k_ids, v_ids}, {(uint16_t*)k_payload, (uint16_t*)v_payload}, {k_meta, v_meta}, {Ck, Cv}};
    if (planes_ok(S, 2) && (rows <= kFewRows16 || T >= kTokensBitmap))
        return launch_planes<false>(S, 2, B, H, T, nnz, (hipStream_t)stream);
    if (reskv_compress_bitmap(k, k_centroids, k_ids, k_payload, k_meta, B, H, T, Ck, nnz, stream)) return 1;
    return reskv_compress_bitmap(v, v_centroids, v_ids, v_payload, v_meta, B, H, T, Cv, nnz, stream);
}
