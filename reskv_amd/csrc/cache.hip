// Small device work of the cache around compression and decode, each one launch in
// the place of a chain of torch kernels whose data takes less time than the gaps.
//
// Ring of recent tokens: one decode token's rotated K, pre-RoPE K and V into their
// slot (three strided copies otherwise).
// Range check of a given clustering's ids, K and V together (comparisons, an or and a
// reduction for each otherwise: 52 us for 2 x 1,048,576 ids, 5 us here).
#include "common.h"
#include "../../include/reskv_hip.h"

using namespace reskv;

namespace {

struct RingArgs {
    const uint4* src[3];   // rows of batch b, head h at b * sb + h * sh
    long sb[3], sh[3];     // in 16-byte units
    uint4* ring[3];        // [B, H, cap, 128] of 2-byte values
    int B, H, cap, slot;
};

// One thread per 16 bytes: 16 per row, rows of the three tensors one after the other.
__global__ void __launch_bounds__(256) ring_append_kernel(RingArgs A) {
    const int rows = A.B * A.H;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    const int row = idx >> 4, piece = idx & 15;
    if (row >= 3 * rows) return;
    const int which = row / rows, bh = row - which * rows;
    const int b = bh / A.H, h = bh - b * A.H;
    // selected by comparisons: indexing the argument arrays by `which` would take them through memory
    const uint4* src = which == 0 ? A.src[0] : which == 1 ? A.src[1] : A.src[2];
    const long sb = which == 0 ? A.sb[0] : which == 1 ? A.sb[1] : A.sb[2];
    const long sh = which == 0 ? A.sh[0] : which == 1 ? A.sh[1] : A.sh[2];
    uint4* ring = which == 0 ? A.ring[0] : which == 1 ? A.ring[1] : A.ring[2];
    ring[((long)bh * A.cap + A.slot) * 16 + piece] = src[b * sb + h * sh + piece];
}

struct IdRange {
    const int32_t* ids[2];
    long n[2];
    int count[2];  // valid ids: [0, count)
    int32_t* flags;
};

// flags[side] becomes 1 when an id of that side is out of range (otherwise untouched).
__global__ void __launch_bounds__(256) ids_in_range_kernel(IdRange A) {
    const int side = blockIdx.y;
    const int32_t* ids = side ? A.ids[1] : A.ids[0];
    const long n = side ? A.n[1] : A.n[0];
    const uint32_t count = (uint32_t)(side ? A.count[1] : A.count[0]);
    const long step = (long)gridDim.x * 256;
    uint32_t bad = 0;
    if (((uintptr_t)ids & 15u) == 0) {
        const int4* quads = reinterpret_cast<const int4*>(ids);
        for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n / 4; i += step) {
            const int4 q = quads[i];
            bad |= (uint32_t)q.x >= count || (uint32_t)q.y >= count || (uint32_t)q.z >= count || (uint32_t)q.w >= count;
        }
        for (long i = n / 4 * 4 + (long)blockIdx.x * 256 + threadIdx.x; i < n; i += step) bad |= (uint32_t)ids[i] >= count;
    } else {
        for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += step) bad |= (uint32_t)ids[i] >= count;
    }
    if (bad) A.flags[side] = 1;
}

}  // namespace

extern "C" int reskv_ids_in_range(const int32_t* k_ids, int64_t nk, int k_count, const int32_t* v_ids, int64_t nv,
                                  int v_count, int32_t* flags, void* stream) {
    RESKV_REQUIRE(k_ids && v_ids && flags, "null pointer argument");
    RESKV_REQUIRE(nk > 0 && nv > 0 && k_count > 0 && v_count > 0, "id and centroid counts must be positive");
    const int64_t most = nk > nv ? nk : nv, blocks = (most + 4095) / 4096;  // 16 ids per thread
    const IdRange A{{k_ids, v_ids}, {(long)nk, (long)nv}, {k_count, v_count}, flags};
    hipLaunchKernelGGL(ids_in_range_kernel, dim3((unsigned)(blocks < 2048 ? blocks : 2048), 2), dim3(256), 0,
                       (hipStream_t)stream, A);
    return reskv_host::check_launch("ids_in_range_kernel");
}

extern "C" int reskv_ring_append(const void* k_rot, const void* k_raw, const void* v, const int64_t* strides,
                                 void* ring_rot, void* ring_raw, void* ring_v, int B, int H, int cap, int slot,
                                 void* stream) {
    RESKV_REQUIRE(k_rot && k_raw && v && strides && ring_rot && ring_raw && ring_v, "null pointer argument");
    RESKV_REQUIRE(B > 0 && H > 0 && cap > 0 && slot >= 0 && slot < cap, "bad ring sizes (B %d, H %d, capacity %d, slot %d)",
                  B, H, cap, slot);
    RESKV_REQUIRE((long)B * H < (1L << 24), "too many (batch, head) rows");
    const void* const src[3] = {k_rot, k_raw, v};
    void* const ring[3] = {ring_rot, ring_raw, ring_v};
    RingArgs A{};
    for (int i = 0; i < 3; ++i) {
        RESKV_REQUIRE((((uintptr_t)src[i] | (uintptr_t)ring[i]) & 15u) == 0 && strides[2 * i] % 8 == 0 &&
                          strides[2 * i + 1] % 8 == 0, "ring append needs 16-byte aligned rows");
        A.src[i] = (const uint4*)src[i];
        A.ring[i] = (uint4*)ring[i];
        A.sb[i] = strides[2 * i] / 8;
        A.sh[i] = strides[2 * i + 1] / 8;
    }
    A.B = B;
    A.H = H;
    A.cap = cap;
    A.slot = slot;
    const int threads = 3 * B * H * 16;
    hipLaunchKernelGGL(ring_append_kernel, dim3((threads + 255) / 256), dim3(256), 0, (hipStream_t)stream, A);
    return reskv_host::check_launch("ring_append_kernel");
}
