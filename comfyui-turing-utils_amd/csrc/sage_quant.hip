// Sage attention prologue for gfx950: K channel mean (smoothing) and
// per-block symmetric INT8 quantization of Q and K.
//
// Quantizer semantics: QuantInt8Kernel (kernel/csrc/turing/sage/fused.cu
// :66-200) with sub_mean (:97-128):
//   v = float(x) - float(mean[d]);  amax = max(1e-7, max|v| over the block)
//   scale = amax / 127;  q = cvt.rni.sat.s8(v * (127 / amax))
// The reference compiles this with --use_fast_math; here both divisions are
// IEEE, as in the CPU oracle.
//
// The K mean is not defined by the reference (its production Sage path has
// smoothing switched off, turing_sage/core.py:421).  This build defines it as
// bf16_rn(sum_t k[t][d] / L) with a fixed fp32 summation order, so that the
// oracle can restate it bit for bit:
//   chunk c = tokens [128c, 128c + 128); a 256-thread workgroup gives each
//   thread 8 channels of every rows-th token (rows = 256 / (D/8));
//   per-thread sums run over ascending tokens, the rows partial sums of a
//   chunk are added in ascending row order, and the chunk sums in ascending
//   chunk order by a second kernel.
#include <mutex>

#include "sage_prep.h"

namespace tu {
namespace {

constexpr int kThreads = 256;

// Chunk-sum scratch of tu_sage_kmean_noalloc: a file-scope device array that
// every GPU running this library holds until the process ends.  In host code
// `scratch` names a host-side stand-in, not a device address; the device
// address comes from hipGetSymbolAddress, once per device (scratch_ptr).
constexpr int64_t kNoAllocScratchFloats = int64_t{1} << 22;  // 16 MiB
static __device__ __align__(256) float scratch[kNoAllocScratchFloats];

template <int D>
__global__ __launch_bounds__(kThreads) void kmean_chunk_kernel(const uint16_t *__restrict__ k, int64_t len,
                                                               int64_t s_b, int64_t s_h, int64_t s_l,
                                                               float *__restrict__ chunk_sums) {
    __shared__ float partial[kThreads / (D / 8)][D];
    kmean_chunk<D>(k, len, s_b, s_h, s_l, chunk_sums, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.y, gridDim.x,
                   partial);
}

// The bf16 mean of one channel: the sum of its chunk sums (dim apart) in
// ascending order, divided by len.  Loads are issued 16 at a time to hide
// their latency; the additions stay in ascending chunk order.
__device__ __forceinline__ uint16_t chunk_mean(const float *__restrict__ src, int64_t chunks, int64_t len, int dim) {
    float tot = 0.0f;
    int64_t c = 0;
    for (; c + 16 <= chunks; c += 16) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) v[j] = src[(c + j) * dim];
#pragma unroll
        for (int j = 0; j < 16; ++j) tot = tot + v[j];
    }
    for (; c < chunks; ++c) tot = tot + src[c * dim];
    return static_cast<uint16_t>(bf16_rne_bits(tot / static_cast<float>(len)));
}

// One thread per (batch*head, channel).
__global__ __launch_bounds__(128) void kmean_final_kernel(const float *__restrict__ chunk_sums, int64_t chunks,
                                                          int64_t len, int dim, uint16_t *__restrict__ mean) {
    const int d = threadIdx.x;
    if (d >= dim) return;
    const int64_t bh = blockIdx.x;
    mean[bh * dim + d] = chunk_mean(chunk_sums + bh * chunks * dim + d, chunks, len, dim);
}

// The means of 8 channels from a bf16 [batch * heads][D] array.
__device__ __forceinline__ void load_means(float (&mu)[8], const uint16_t *mean) {
    const u32x4 mv = *reinterpret_cast<const u32x4 *>(mean);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        mu[2 * e] = bf16_bits_to_f32(mv[e] & 0xffffu);
        mu[2 * e + 1] = bf16_bits_to_f32(mv[e] >> 16);
    }
}

template <int D, int BLK, bool kSubMean>
__global__ __launch_bounds__(kThreads) void sage_quant_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ mean, int64_t len, int64_t s_b,
    int64_t s_h, int64_t s_l, int8_t *__restrict__ q, int64_t q_b, int64_t q_h, int64_t q_l,
    float *__restrict__ scale) {
    __shared__ float wave_amax[kThreads / 64];
    const int64_t h = blockIdx.y, b = blockIdx.z, heads = gridDim.y;
    auto means = [&](float (&mu)[8], int c8) { load_means(mu, mean + (b * heads + h) * D + c8 * 8); };
    quant_block<D, BLK, kSubMean>(x, means, len, s_b, s_h, s_l, q, q_b, q_h, q_l, scale, blockIdx.x, h, b, heads,
                                  gridDim.x, wave_amax);
}

template <int D>
int32_t launch_quant(const uint16_t *x, const uint16_t *mean, int64_t batch, int64_t heads, int64_t len,
                     int64_t s_b, int64_t s_h, int64_t s_l, int64_t blk, int8_t *q, int64_t q_b, int64_t q_h,
                     int64_t q_l, float *scale, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>((len + blk - 1) / blk), static_cast<unsigned>(heads),
                    static_cast<unsigned>(batch));
#define TU_QUANT_CASE(B)                                                                                \
    case B:                                                                                             \
        if (mean)                                                                                       \
            sage_quant_kernel<D, B, true><<<grid, kThreads, 0, s>>>(x, mean, len, s_b, s_h, s_l, q, q_b, \
                                                                    q_h, q_l, scale);                   \
        else                                                                                            \
            sage_quant_kernel<D, B, false><<<grid, kThreads, 0, s>>>(x, mean, len, s_b, s_h, s_l, q,     \
                                                                     q_b, q_h, q_l, scale);             \
        break;
    switch (blk) {
        TU_QUANT_CASE(16)
        TU_QUANT_CASE(32)
        TU_QUANT_CASE(64)
        TU_QUANT_CASE(128)
        default:
            return fail("Sage quantization block must be 16, 32, 64 or 128, got %lld", static_cast<long long>(blk));
    }
#undef TU_QUANT_CASE
    return check_launch("tu_sage_quant");
}

// ---------------------------------------------------------------------------
// The whole prologue of a Sage attention call in two launches (three past 64
// K chunks).  As five kernels, each with a ramp, a tail and a launch of its
// own, it took 42 us at B1 H12 L8190 D128 for 113 MB of traffic that a copy
// moves in about 20, and 16 us for a call of 300 tokens; now 38 and 9 us.  Q's blocks, V's tiles
// and K's chunk sums depend on nothing, so they share one grid; K's blocks,
// which need K's mean, follow.  With at most kInlineChunks chunk sums a head
// every K block adds them itself (in kmean_final_kernel's order, so the mean
// has the same bits); past that a block would read more sums than tokens and
// the mean has its launch.
// ---------------------------------------------------------------------------
constexpr int64_t kInlineChunks = 64;

struct PrepArgs {
    const uint16_t *q, *k, *v;
    int64_t lq, lk, lpad;
    int64_t q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, v_sb, v_sh, v_sl;
    int8_t *q8, *k8;
    int64_t q8_sb, q8_sh, q8_sl, k8_sb, k8_sh, k8_sl;
    float *q_scale, *k_scale;
    uint16_t *vt;
    float *chunk_sums;
    uint16_t *mean;
    uint32_t batch, hq, hkv;
    uint32_t q_blocks, v_tiles, k_chunks, k_blocks;  // of one head
};

// Workgroups: V tiles, then K chunks (kSmooth), then Q blocks; each block
// fastest, then head, then batch.
template <int D, int BLKQ, bool kSmooth>
__global__ __launch_bounds__(kPrepThreads) void sage_prep_kernel(PrepArgs a) {
    __shared__ union {
        uint16_t tile[kPrepKeys][D + 4];
        float partial[kPrepThreads / (D / 8)][D];
        float wave_amax[kPrepThreads / 64];
    } lds;
    uint32_t id = blockIdx.x;
    const uint32_t v_wgs = a.v_tiles * a.hkv * a.batch, k_wgs = kSmooth ? a.k_chunks * a.hkv * a.batch : 0;
    if (id < v_wgs) {
        const uint32_t bh = id / a.v_tiles;
        v_prep_tile<D>(a.v, a.lk, a.lpad, a.v_sb, a.v_sh, a.v_sl, a.vt, id % a.v_tiles, bh % a.hkv, bh / a.hkv, a.hkv,
                       lds.tile);
        return;
    }
    id -= v_wgs;
    if (kSmooth && id < k_wgs) {
        const uint32_t bh = id / a.k_chunks;
        kmean_chunk<D>(a.k, a.lk, a.k_sb, a.k_sh, a.k_sl, a.chunk_sums, id % a.k_chunks, bh % a.hkv, bh / a.hkv, a.hkv,
                       a.k_chunks, lds.partial);
        return;
    }
    id -= k_wgs;
    const uint32_t bh = id / a.q_blocks;
    quant_block<D, BLKQ, false>(a.q, [](float (&)[8], int) {}, a.lq, a.q_sb, a.q_sh, a.q_sl, a.q8, a.q8_sb, a.q8_sh,
                                a.q8_sl, a.q_scale, id % a.q_blocks, bh % a.hq, bh / a.hq, a.hq, a.q_blocks,
                                lds.wave_amax);
}

// K blocks.  kMean: 0 no smoothing, 1 the mean from a.mean, 2 from the chunk sums.
template <int D, int BLKK, int kMean>
__global__ __launch_bounds__(kPrepThreads) void sage_prep_k_kernel(PrepArgs a) {
    __shared__ float wave_amax[kPrepThreads / 64];
    __shared__ __align__(16) uint16_t mean[D];
    const uint32_t blk = blockIdx.x % a.k_blocks, bh = blockIdx.x / a.k_blocks;
    if constexpr (kMean == 2) {
        const int d = threadIdx.x;
        if (d < D) mean[d] = chunk_mean(a.chunk_sums + static_cast<int64_t>(bh) * a.k_chunks * D + d, a.k_chunks, a.lk, D);
        __syncthreads();
    }
    auto means = [&](float (&mu)[8], int c8) {
        load_means(mu, kMean == 2 ? mean + c8 * 8 : a.mean + static_cast<int64_t>(bh) * D + c8 * 8);
    };
    quant_block<D, BLKK, kMean != 0>(a.k, means, a.lk, a.k_sb, a.k_sh, a.k_sl, a.k8, a.k8_sb, a.k8_sh, a.k8_sl,
                                     a.k_scale, blk, bh % a.hkv, bh / a.hkv, a.hkv, a.k_blocks, wave_amax);
}

template <int D>
int32_t launch_prep(const PrepArgs &a, int64_t blkq, int64_t blkk, bool smooth, hipStream_t s) {
    const dim3 grid1(a.batch * (a.v_tiles * a.hkv + (smooth ? a.k_chunks * a.hkv : 0) + a.q_blocks * a.hq));
#define TU_PREP_CASE(B)                                                                  \
    case B:                                                                              \
        if (smooth) sage_prep_kernel<D, B, true><<<grid1, kPrepThreads, 0, s>>>(a);       \
        else sage_prep_kernel<D, B, false><<<grid1, kPrepThreads, 0, s>>>(a);             \
        break;
    switch (blkq) {
        TU_PREP_CASE(16)
        TU_PREP_CASE(32)
        TU_PREP_CASE(64)
        TU_PREP_CASE(128)
        default: return fail("Sage quantization block must be 16, 32, 64 or 128, got %lld", static_cast<long long>(blkq));
    }
#undef TU_PREP_CASE
    if (check_launch("tu_sage_prep")) return -1;
    const bool inline_mean = smooth && a.k_chunks <= kInlineChunks;
    if (smooth && !inline_mean) {
        kmean_final_kernel<<<dim3(a.batch * a.hkv), 128, 0, s>>>(a.chunk_sums, a.k_chunks, a.lk, D, a.mean);
        if (check_launch("tu_sage_prep(mean)")) return -1;
    }
    const dim3 grid2(a.batch * a.hkv * a.k_blocks);
#define TU_PREP_CASE(B)                                                                        \
    case B:                                                                                    \
        if (!smooth) sage_prep_k_kernel<D, B, 0><<<grid2, kPrepThreads, 0, s>>>(a);             \
        else if (!inline_mean) sage_prep_k_kernel<D, B, 1><<<grid2, kPrepThreads, 0, s>>>(a);   \
        else sage_prep_k_kernel<D, B, 2><<<grid2, kPrepThreads, 0, s>>>(a);                     \
        break;
    switch (blkk) {
        TU_PREP_CASE(64)
        TU_PREP_CASE(128)
        default: return fail("Sage K block must be 64 or 128, got %lld", static_cast<long long>(blkk));
    }
#undef TU_PREP_CASE
    return check_launch("tu_sage_prep(K)");
}

}  // namespace
}  // namespace tu

extern "C" int32_t tu_sage_kmean(const void *k_bf16, int64_t batch, int64_t heads, int64_t len, int64_t dim,
                                 int64_t s_b, int64_t s_h, int64_t s_l, float *chunk_sums, void *mean_bf16,
                                 void *stream) {
    using namespace tu;
    TU_REQUIRE(dim == 64 || dim == 128, "K mean requires head_dim 64 or 128, got %lld", static_cast<long long>(dim));
    TU_REQUIRE(batch > 0 && heads > 0 && len > 0, "K mean requires positive batch, heads and length");
    TU_REQUIRE(heads <= 65535 && batch <= 65535 && (len + 127) / 128 <= 0x7fffffff, "K mean grid too large");
    TU_REQUIRE(k_bf16 && chunk_sums && mean_bf16, "K mean pointers must be non-null");
    TU_REQUIRE(s_l % 8 == 0 && s_h % 8 == 0 && s_b % 8 == 0 && (reinterpret_cast<uintptr_t>(k_bf16) & 15) == 0,
               "K mean needs 16-byte aligned token rows");
    if (require_gfx950()) return -1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t chunks = (len + 127) / 128;
    const dim3 grid(static_cast<unsigned>(chunks), static_cast<unsigned>(heads), static_cast<unsigned>(batch));
    const auto *k = static_cast<const uint16_t *>(k_bf16);
    if (dim == 128) kmean_chunk_kernel<128><<<grid, kThreads, 0, s>>>(k, len, s_b, s_h, s_l, chunk_sums);
    else kmean_chunk_kernel<64><<<grid, kThreads, 0, s>>>(k, len, s_b, s_h, s_l, chunk_sums);
    if (check_launch("tu_sage_kmean(chunks)")) return -1;
    kmean_final_kernel<<<dim3(static_cast<unsigned>(batch * heads)), 128, 0, s>>>(
        chunk_sums, chunks, len, static_cast<int>(dim), static_cast<uint16_t *>(mean_bf16));
    return check_launch("tu_sage_kmean(final)");
}

namespace tu {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float *g_scratch_ptr[kMaxDevices];

// Device address of `scratch` on the current device, looked up on the first
// call on that device (with the device current) and kept per device.
int32_t scratch_ptr(float **out) {
    int dev = 0;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return fail("hipGetDevice failed: %s", hipGetErrorString(err));
    if (dev < 0 || dev >= kMaxDevices) return fail("device %d is beyond the %d devices this library serves", dev,
                                                   kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !p)
            return fail("hipGetSymbolAddress(scratch) on device %d failed: %s", dev, hipGetErrorString(err));
        g_scratch_ptr[dev] = static_cast<float *>(p);
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

}  // namespace
}  // namespace tu

extern "C" int32_t tu_sage_kmean_noalloc(const void *k_bf16, int64_t batch, int64_t heads, int64_t len,
                                         int64_t dim, int64_t s_b, int64_t s_h, int64_t s_l, void *mean_bf16,
                                         void *stream) {
    using namespace tu;
    TU_REQUIRE(dim == 64 || dim == 128, "K mean requires head_dim 64 or 128, got %lld", static_cast<long long>(dim));
    TU_REQUIRE(batch > 0 && heads > 0 && len > 0, "K mean requires positive batch, heads and length");
    TU_REQUIRE(heads <= 65535 && batch <= 65535 && (len + 127) / 128 <= 0x7fffffff, "K mean grid too large");
    TU_REQUIRE(k_bf16 && mean_bf16, "K mean pointers must be non-null");
    TU_REQUIRE(s_l % 8 == 0 && s_h % 8 == 0 && s_b % 8 == 0 && (reinterpret_cast<uintptr_t>(k_bf16) & 15) == 0,
               "K mean needs 16-byte aligned token rows");
    const int64_t chunks = (len + 127) / 128;
    // batch, heads <= 65535 and chunks < 2^31 cannot overflow the product in
    // steps: check each factor against the limit first
    TU_REQUIRE(chunks <= kNoAllocScratchFloats / dim &&
                   batch * heads <= kNoAllocScratchFloats / (chunks * dim),
               "K mean without allocation: batch*heads*ceil(len/128)*dim = %lld*%lld*%lld*%lld exceeds the "
               "%lld-float scratch (use tu_sage_kmean with caller scratch)",
               static_cast<long long>(batch), static_cast<long long>(heads), static_cast<long long>(chunks),
               static_cast<long long>(dim), static_cast<long long>(kNoAllocScratchFloats));
    if (require_gfx950()) return -1;
    float *chunk_sums = nullptr;
    if (scratch_ptr(&chunk_sums)) return -1;
    // Every chunk sum the final kernel reads is written by the chunk kernel
    // of the same call first, so nothing needs clearing.
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>(chunks), static_cast<unsigned>(heads), static_cast<unsigned>(batch));
    const auto *k = static_cast<const uint16_t *>(k_bf16);
    if (dim == 128) kmean_chunk_kernel<128><<<grid, kThreads, 0, s>>>(k, len, s_b, s_h, s_l, chunk_sums);
    else kmean_chunk_kernel<64><<<grid, kThreads, 0, s>>>(k, len, s_b, s_h, s_l, chunk_sums);
    if (check_launch("tu_sage_kmean_noalloc(chunks)")) return -1;
    kmean_final_kernel<<<dim3(static_cast<unsigned>(batch * heads)), 128, 0, s>>>(
        chunk_sums, chunks, len, static_cast<int>(dim), static_cast<uint16_t *>(mean_bf16));
    return check_launch("tu_sage_kmean_noalloc(final)");
}

extern "C" int32_t tu_sage_quant(const void *x_bf16, const void *mean_bf16, int64_t batch, int64_t heads,
                                 int64_t len, int64_t dim, int64_t s_b, int64_t s_h, int64_t s_l, int64_t blk,
                                 int8_t *q, int64_t q_b, int64_t q_h, int64_t q_l, float *scale, void *stream) {
    using namespace tu;
    TU_REQUIRE(dim == 64 || dim == 128, "Sage quantization requires head_dim 64 or 128, got %lld",
               static_cast<long long>(dim));
    TU_REQUIRE(batch > 0 && heads > 0 && len > 0, "Sage quantization requires positive batch, heads and length");
    TU_REQUIRE(heads <= 65535 && batch <= 65535, "Sage quantization grid too large");
    TU_REQUIRE(x_bf16 && q && scale, "Sage quantization pointers must be non-null");
    TU_REQUIRE(s_l % 8 == 0 && s_h % 8 == 0 && s_b % 8 == 0 && (reinterpret_cast<uintptr_t>(x_bf16) & 15) == 0,
               "Sage quantization needs 16-byte aligned token rows");
    TU_REQUIRE(q_l % 8 == 0 && q_h % 8 == 0 && q_b % 8 == 0 && (reinterpret_cast<uintptr_t>(q) & 7) == 0,
               "Sage quantization output needs 8-byte aligned token rows");
    TU_REQUIRE(!mean_bf16 || (reinterpret_cast<uintptr_t>(mean_bf16) & 15) == 0, "K mean must be 16-byte aligned");
    if (require_gfx950()) return -1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const auto *x = static_cast<const uint16_t *>(x_bf16);
    const auto *mean = static_cast<const uint16_t *>(mean_bf16);
    if (dim == 128) return launch_quant<128>(x, mean, batch, heads, len, s_b, s_h, s_l, blk, q, q_b, q_h, q_l, scale, s);
    return launch_quant<64>(x, mean, batch, heads, len, s_b, s_h, s_l, blk, q, q_b, q_h, q_l, scale, s);
}

extern "C" int64_t tu_sage_prep_workspace(int64_t batch, int64_t hkv, int64_t lk, int64_t dim, int32_t smooth_k) {
    if (!smooth_k || batch <= 0 || hkv <= 0 || lk <= 0 || dim <= 0) return 0;
    const int64_t chunks = (lk + 127) / 128;
    // chunk sums, then (past the inline limit) the bf16 means
    return batch * hkv * dim * (chunks * 4 + (chunks > tu::kInlineChunks ? 2 : 0));
}

extern "C" int32_t tu_sage_prep(const void *q_bf16, const void *k_bf16, const void *v_bf16, int64_t batch, int64_t hq,
                                int64_t hkv, int64_t lq, int64_t lk, int64_t dim, int64_t q_sb, int64_t q_sh,
                                int64_t q_sl, int64_t k_sb, int64_t k_sh, int64_t k_sl, int64_t v_sb, int64_t v_sh,
                                int64_t v_sl, int32_t smooth_k, int64_t blkq, int64_t blkk, int8_t *q8, int64_t q8_sb,
                                int64_t q8_sh, int64_t q8_sl, int8_t *k8, int64_t k8_sb, int64_t k8_sh, int64_t k8_sl,
                                float *q_scale, float *k_scale, void *vt_bf16, int64_t lpad, void *workspace,
                                int64_t workspace_bytes, void *stream) {
    using namespace tu;
    TU_REQUIRE(dim == 64 || dim == 128, "Sage prologue requires head_dim 64 or 128, got %lld",
               static_cast<long long>(dim));
    TU_REQUIRE(batch > 0 && hq > 0 && hkv > 0 && lq > 0 && lk > 0,
               "Sage prologue requires positive batch, heads and lengths");
    TU_REQUIRE(lpad >= lk && lpad % kPrepKeys == 0, "V^T padded length must cover lk and be a multiple of 64");
    TU_REQUIRE((blkq == 16 || blkq == 32 || blkq == 64 || blkq == 128) && (blkk == 64 || blkk == 128),
               "Sage prologue blocks must be 16 to 128 (Q) and 64 or 128 (K), got %lld and %lld",
               static_cast<long long>(blkq), static_cast<long long>(blkk));
    TU_REQUIRE(q_bf16 && k_bf16 && v_bf16 && q8 && k8 && q_scale && k_scale && vt_bf16,
               "Sage prologue pointers must be non-null");
    auto aligned = [](const void *p, int64_t sb, int64_t sh, int64_t sl, uintptr_t bytes) {
        return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0 && sb % 8 == 0 && sh % 8 == 0 && sl % 8 == 0;
    };
    TU_REQUIRE(aligned(q_bf16, q_sb, q_sh, q_sl, 16) && aligned(k_bf16, k_sb, k_sh, k_sl, 16) &&
                   aligned(v_bf16, v_sb, v_sh, v_sl, 16) && aligned(vt_bf16, 0, 0, 0, 16),
               "Sage prologue needs 16-byte aligned token rows");
    TU_REQUIRE(aligned(q8, q8_sb, q8_sh, q8_sl, 8) && aligned(k8, k8_sb, k8_sh, k8_sl, 8),
               "Sage prologue output needs 8-byte aligned token rows");
    const int64_t need = tu_sage_prep_workspace(batch, hkv, lk, dim, smooth_k);
    TU_REQUIRE(need == 0 || (workspace && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0 && workspace_bytes >= need),
               "Sage prologue workspace must be 16-byte aligned and hold %lld bytes", static_cast<long long>(need));
    const int64_t chunks = (lk + 127) / 128, q_blocks = (lq + blkq - 1) / blkq, k_blocks = (lk + blkk - 1) / blkk;
    // heads and batch as in the separate entry points; every grid, and so every
    // part of one, below 2^23 workgroups (2^31 threads)
    constexpr int64_t kMost = int64_t{1} << 23;
    TU_REQUIRE(batch <= 65535 && hq <= 65535 && hkv <= 65535 && q_blocks <= kMost && lpad / kPrepKeys <= kMost &&
                   batch * hkv <= kMost && batch * hq <= kMost &&
                   batch * (hkv * (lpad / kPrepKeys + chunks) + hq * q_blocks) <= kMost && batch * hkv * k_blocks <= kMost,
               "Sage prologue grid too large");
    if (require_gfx950()) return -1;
    PrepArgs a;
    a.q = static_cast<const uint16_t *>(q_bf16);
    a.k = static_cast<const uint16_t *>(k_bf16);
    a.v = static_cast<const uint16_t *>(v_bf16);
    a.lq = lq, a.lk = lk, a.lpad = lpad;
    a.q_sb = q_sb, a.q_sh = q_sh, a.q_sl = q_sl, a.k_sb = k_sb, a.k_sh = k_sh, a.k_sl = k_sl;
    a.v_sb = v_sb, a.v_sh = v_sh, a.v_sl = v_sl;
    a.q8 = q8, a.q8_sb = q8_sb, a.q8_sh = q8_sh, a.q8_sl = q8_sl;
    a.k8 = k8, a.k8_sb = k8_sb, a.k8_sh = k8_sh, a.k8_sl = k8_sl;
    a.q_scale = q_scale, a.k_scale = k_scale, a.vt = static_cast<uint16_t *>(vt_bf16);
    a.chunk_sums = static_cast<float *>(workspace);
    a.mean = reinterpret_cast<uint16_t *>(a.chunk_sums + batch * hkv * chunks * dim);
    a.batch = static_cast<uint32_t>(batch), a.hq = static_cast<uint32_t>(hq), a.hkv = static_cast<uint32_t>(hkv);
    a.q_blocks = static_cast<uint32_t>(q_blocks), a.v_tiles = static_cast<uint32_t>(lpad / kPrepKeys);
    a.k_chunks = static_cast<uint32_t>(chunks), a.k_blocks = static_cast<uint32_t>(k_blocks);
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dim == 128 ? launch_prep<128>(a, blkq, blkk, smooth_k != 0, s) : launch_prep<64>(a, blkq, blkk, smooth_k != 0, s);
}
