// Prompt pass of the end-to-end decoder (reskv_amd/llama.py): the split / rotation
// of a prompt's Q, K and V, and causal attention over it.
//
// Attention: one workgroup of four waves per 128 (query, head) rows of one KV
// head, a wave owning 32 queries of one query head; the query heads of a KV head
// share the staged K and V.  Keys are taken 64 at a time from double-buffered LDS.
//   S^T = K Q^T on v_mfma_f32_32x32x16_f16: lane (col = lane % 32, half = lane / 32)
//     holds its query's scores of keys 8 (i / 4) + 4 half + i % 4, i = 0..15, of a
//     32-key block, so the softmax needs one lane swap, and the fp16 weights are the
//     B operand of
//   O^T = V^T P^T as they are: its 16-key steps take the keys in the order in which
//     a lane holds them, and V^T comes from the staged rows through LDS transpose
//     reads of the same keys.
// Scores, softmax and sums are fp32; the weights (not larger than 1) are rounded to
// fp16 for the second product and divided by their fp32 sum at the end.
#include "common.h"
#include "reskv_llama.h"

using namespace reskv;

namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) short4_t lds_short4_t;

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * kWave;
constexpr int kQ = 32;             // queries per wave
constexpr int kKeys = 64;          // keys per tile
constexpr int kPitch = kDim + 8;   // halves per staged row (16-byte aligned, rows start on different banks)
constexpr int kTileHalves = kKeys * kPitch;
constexpr int kPieces = kKeys * kDim / 8 / kThreads;  // 16-byte pieces of a K (or V) tile per thread

struct AttnArgs {
    const uint16_t* q;  // [B, Hq, T, 128], rotated
    const uint16_t* k;  // [B, Hk, T, 128], rotated
    const uint16_t* v;  // [B, Hk, T, 128]
    uint16_t* out;      // [B, T, Hq, 128]
    int Hq, Hk, T, pairs;  // pairs: (batch, KV head, group of HPW query heads)
    float c;               // scaling * log2(e)
};

// HPW: query heads of the workgroup (4 / HPW blocks of 32 queries each).
//
// Bound: matrix cores and LDS together.  A wave issues 32 products of 32 cycles per
// tile and reads 32 KB of LDS, and four waves of a CU's two workgroups share 128
// bytes a cycle of it, so both take about 1024 cycles; the softmax of the other
// workgroup runs beside them.  32 / 8 heads, one prompt, back to back: 1024 tokens 31 us,
// 4096 179 us (768 TFLOP/s over the causal half), 8192 632 us (869 TFLOP/s), and 230 us at
// 4096 within a prompt pass, after the projections; in torch (two
// matrix products with fp32 scores, mask and softmax passes between them) a prompt of
// 4096 took about 4 ms.
template <int HPW>
__global__ void __launch_bounds__(kThreads, 2) prefill_attention_kernel(AttnArgs A) {
    constexpr int QB = kWaves / HPW;
    __shared__ __align__(16) uint16_t s_kv[2][2][kTileHalves];  // [buffer][K, V]
    // heaviest query tiles first; consecutive workgroups take the pairs in turn, so
    // that a pair's workgroups share an XCD's L2 when there is a multiple of 8 of them
    const int tiles = (A.T + kQ * QB - 1) / (kQ * QB);
    const int qt = tiles - 1 - (int)blockIdx.x / A.pairs, pair = (int)blockIdx.x % A.pairs;
    const int G = A.Hq / A.Hk, hgs = G / HPW;
    const int hg = pair % hgs, hk = (pair / hgs) % A.Hk;
    const long b = pair / (hgs * A.Hk);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int head = hk * G + hg * HPW + wave % HPW;
    const int q0 = qt * kQ * QB + kQ * (wave / HPW);  // first query of the wave
    const int query = q0 + col;
    const uint16_t* kb = A.k + (b * A.Hk + hk) * (long)A.T * kDim;
    const uint16_t* vb = A.v + (b * A.Hk + hk) * (long)A.T * kDim;

    // Q operand: lane (col, half) holds query col, channels 16 kk + 8 half + [0, 8)
    half8_t qf[8];
    {
        const int row = query < A.T ? query : A.T - 1;
        const uint4* src = reinterpret_cast<const uint4*>(A.q + ((b * A.Hq + head) * (long)A.T + row) * kDim);
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) qf[kk] = __builtin_bit_cast(half8_t, src[2 * kk + half]);
    }

    const int last = min(A.T, (qt + 1) * kQ * QB);  // keys of the workgroup's last query
    const int ntiles = (last + kKeys - 1) / kKeys;
    // Tiles are fetched through range-checked buffer loads without branches (past the
    // last row they return zeros), so that the rows stay in registers while in flight.
    const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc((void*)kb, 0, A.T * kDim * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc((void*)vb, 0, A.T * kDim * 2, 0x00020000);
    uint4 kr[kPieces], vr[kPieces];
    auto fetch = [&](int tile) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int off = tile * (kKeys * kDim * 2) + 16 * (tid + kThreads * i);
            kr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kres, off, 0, 0));
            vr[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vres, off, 0, 0));
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int p = tid + kThreads * i;
            const int at = (p >> 4) * kPitch + 8 * (p & 15);
            *reinterpret_cast<uint4*>(&s_kv[buf][0][at]) = kr[i];
            *reinterpret_cast<uint4*>(&s_kv[buf][1][at]) = vr[i];
        }
    };
    fetch(0);
    stage(0);
    __syncthreads();

    float16_t acc[4];  // O^T: channels 32 db + 8 (i / 4) + 4 half + i % 4 of the lane's query
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[db][i] = 0.0f;
    // log2-domain maximum, and this lane's half of the weights' sum.  The maximum starts at
    // the lowest finite value: scores of minus infinity then weigh exp2(-inf) = 0, where
    // against a maximum of minus infinity they would give NaN
    float m = -__FLT_MAX__, l = 0.0f;
    // transpose reads: lane i of a 16-lane row points at key i / 4, channel 4 (i % 4) of
    // its 4 x 16 block and receives the block's four keys of channel i
    const int i16 = lane & 15;
    const int vt = (4 * half + (i16 >> 2)) * kPitch + 16 * ((lane >> 4) & 1) + 4 * (i16 & 3);

    for (int tile = 0; tile < ntiles; ++tile) {
        const int buf = tile & 1, base = tile * kKeys;
        fetch(tile + 1);
        if (base <= q0 + kQ - 1) {  // wave-uniform: a tile past the wave's queries is left out
            const uint16_t* sk = s_kv[buf][0];
            const uint16_t* sv = s_kv[buf][1];
            float16_t s[2];
#pragma unroll
            for (int kb2 = 0; kb2 < 2; ++kb2) {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[kb2][i] = 0.0f;
#pragma unroll
                for (int kk = 0; kk < 8; ++kk) {
                    const half8_t kf = *reinterpret_cast<const half8_t*>(sk + (32 * kb2 + col) * kPitch + 16 * kk + 8 * half);
                    s[kb2] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[kk], s[kb2], 0, 0, 0);
                }
            }
            if (base + kKeys - 1 > q0) {  // the diagonal
#pragma unroll
                for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (base + 32 * kb2 + 8 * (i >> 2) + 4 * half + (i & 3) > query) s[kb2][i] = -INFINITY;
            }
            float mx = s[0][0];
#pragma unroll
            for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
                for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kb2][i]);
            const auto sw = __builtin_amdgcn_permlane32_swap((uint32_t)f2i(mx), (uint32_t)f2i(mx), false, false);
            mx = fmaxf(i2f((int)sw[0]), i2f((int)sw[1])) * A.c;  // c > 0
            if (ballot(mx > m) != 0) {
                const float mn = fmaxf(m, mx);
                const float alpha = __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                l *= alpha;
#pragma unroll
                for (int db = 0; db < 4; ++db)
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[db][i] *= alpha;
            }
            half8_t pf[4];  // the weights of 16-key steps, keys in the lane's order
            float sum = 0.0f;
#pragma unroll
            for (int kb2 = 0; kb2 < 2; ++kb2)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb2][i], A.c, -m));
                    sum += p;
                    pf[2 * kb2 + (i >> 3)][i & 7] = (_Float16)p;
                }
            l += sum;
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int db = 0; db < 4; ++db) {
                    const uint16_t* src = sv + vt + 16 * st * kPitch + 32 * db;
                    const half4_t lo = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)src));
                    const half4_t hi = __builtin_bit_cast(
                        half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)(src + 8 * kPitch)));
                    const half8_t vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                    acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[st], acc[db], 0, 0, 0);
                }
        }
        stage(buf ^ 1);  // last read in the tile before, which a barrier ended
        __syncthreads();
    }

    const auto ls = __builtin_amdgcn_permlane32_swap((uint32_t)f2i(l), (uint32_t)f2i(l), false, false);
    const float inv = 1.0f / (i2f((int)ls[0]) + i2f((int)ls[1]));
    if (query >= A.T) return;
    uint16_t* dst = A.out + ((b * A.T + query) * A.Hq + head) * kDim;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t w[2];
#pragma unroll
            for (int e = 0; e < 2; ++e)
                w[e] = (uint32_t)f2h(acc[db][4 * j + 2 * e] * inv) | ((uint32_t)f2h(acc[db][4 * j + 2 * e + 1] * inv) << 16);
            *reinterpret_cast<uint2*>(dst + 32 * db + 8 * j + 4 * half) = make_uint2(w[0], w[1]);
        }
}

struct SplitArgs {
    const uint16_t* qkv;  // [B, T, (Hq + 2 Hk) * 128]
    const float* cos;     // [T, 64]
    const float* sin;
    uint16_t *qr, *k, *kr, *v;  // [B, heads, T, 128]
    int T, Hq, Hk;
    long items;  // B * T * (Hq + 2 Hk) * 8
};

// One thread per eight rotate-half pairs (channels 8 j .. 8 j + 7 and those + 64) of one
// head of one token, products and sums rounded as in qkv_rope_kernel.
__global__ void __launch_bounds__(256) prefill_split_kernel(SplitArgs A) {
#pragma clang fp contract(off)  // products and sums rounded apart
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= A.items) return;
    const int heads = A.Hq + 2 * A.Hk;
    const int j = (int)(idx & 7);
    const long row = (idx >> 3) / heads;  // b * T + t
    const int h = (int)((idx >> 3) - row * heads);
    const long b = row / A.T;
    const long t = row - b * A.T;
    const uint4* src = reinterpret_cast<const uint4*>(A.qkv + (row * heads + h) * kDim) + j;
    const uint4 lo = src[0], hi = src[8];
    if (h >= A.Hq + A.Hk) {
        uint4* dv = reinterpret_cast<uint4*>(A.v + ((b * A.Hk + h - A.Hq - A.Hk) * A.T + t) * kDim) + j;
        dv[0] = lo;
        dv[8] = hi;
        return;
    }
    const float4* cp = reinterpret_cast<const float4*>(A.cos + t * kHalf) + 2 * j;
    const float4* sp = reinterpret_cast<const float4*>(A.sin + t * kHalf) + 2 * j;
    const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
    const float c[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
    const float s[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    const uint32_t lw[4] = {lo.x, lo.y, lo.z, lo.w}, hw[4] = {hi.x, hi.y, hi.z, hi.w};
    uint32_t rl[4], rh[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        rl[i] = rh[i] = 0;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float a = h2f((uint16_t)(lw[i] >> (16 * e))), x = h2f((uint16_t)(hw[i] >> (16 * e)));
            const float cc = c[2 * i + e], ss = s[2 * i + e];
            const float ac = a * cc, xs = x * ss, xc = x * cc, as = a * ss;
            rl[i] |= (uint32_t)f2h(ac - xs) << (16 * e);
            rh[i] |= (uint32_t)f2h(xc + as) << (16 * e);
        }
    }
    const uint4 ro = make_uint4(rl[0], rl[1], rl[2], rl[3]), rp = make_uint4(rh[0], rh[1], rh[2], rh[3]);
    if (h < A.Hq) {
        uint4* dq = reinterpret_cast<uint4*>(A.qr + ((b * A.Hq + h) * A.T + t) * kDim) + j;
        dq[0] = ro;
        dq[8] = rp;
        return;
    }
    const long at = ((b * A.Hk + h - A.Hq) * A.T + t) * kDim;
    uint4* dk = reinterpret_cast<uint4*>(A.k + at) + j;
    uint4* dr = reinterpret_cast<uint4*>(A.kr + at) + j;
    dk[0] = lo;
    dk[8] = hi;
    dr[0] = ro;
    dr[8] = rp;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

extern "C" int reskv_llama_prefill_attention(const void* q, const void* k, const void* v, void* out, int B, int Hq,
                                             int Hk, int T, float scaling, void* stream) {
    RESKV_REQUIRE(q && k && v && out, "null pointer");
    RESKV_REQUIRE(B > 0 && T > 0 && Hk > 0 && Hq > 0 && Hq % Hk == 0, "bad sizes (B %d, Hq %d, Hk %d, T %d)", B, Hq, Hk, T);
    const int G = Hq / Hk;
    RESKV_REQUIRE(G == 1 || G == 2 || G % 4 == 0, "the query/KV head ratio %d must be 1, 2 or a multiple of 4", G);
    RESKV_REQUIRE(scaling > 0.0f, "scaling must be positive");
    RESKV_REQUIRE(T <= (1 << 22), "T must not exceed %d (32-bit offsets into a head's rows)", 1 << 22);
    RESKV_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), "tensors must be 16-byte aligned");
    const int hpw = G % 4 == 0 ? 4 : G;
    const long pairs = (long)B * Hk * (G / hpw), tiles = (T + kQ * (kWaves / hpw) - 1) / (kQ * (kWaves / hpw));
    RESKV_REQUIRE(pairs * tiles < (1L << 31), "too many query tiles");
    const AttnArgs A{(const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)out, Hq, Hk, T, (int)pairs,
                     scaling * 1.4426950408889634f};
    const auto kernel = hpw == 4 ? prefill_attention_kernel<4> : hpw == 2 ? prefill_attention_kernel<2> : prefill_attention_kernel<1>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(pairs * tiles)), dim3(kThreads), 0, (hipStream_t)stream, A);
    return reskv_host::check_launch("prefill_attention_kernel");
}

extern "C" int reskv_llama_prefill_split(const void* qkv, const float* cos, const float* sin, int B, int T, int Hq,
                                         int Hk, void* qr, void* k, void* kr, void* v, void* stream) {
    RESKV_REQUIRE(qkv && cos && sin && qr && k && kr && v, "null pointer");
    RESKV_REQUIRE(B > 0 && T > 0 && Hk > 0 && Hq > 0, "sizes must be positive");
    RESKV_REQUIRE(aligned16(qkv) && aligned16(cos) && aligned16(sin) && aligned16(qr) && aligned16(k) && aligned16(kr) &&
                      aligned16(v), "tensors must be 16-byte aligned");
    const long items = (long)B * T * (Hq + 2 * Hk) * 8;
    RESKV_REQUIRE((items + 255) / 256 < (1L << 31), "too many tokens");
    const SplitArgs A{(const uint16_t*)qkv, cos, sin, (uint16_t*)qr, (uint16_t*)k, (uint16_t*)kr, (uint16_t*)v, T, Hq, Hk,
                      items};
    hipLaunchKernelGGL(prefill_split_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, (hipStream_t)stream, A);
    return reskv_host::check_launch("prefill_split_kernel");
}
