// Prologue of the dense W8A8 attention for gfx950: K stabilisation anchor,
// Hadamard-rotated per-tile INT8 Q/K, and channel-wise INT8 V.
//
// Reference semantics (kernel/csrc/turing/sage/):
//   anchor  DetectKAnchorKernel (fused.cu:409-575): nine keys at rows
//           s (L - 1) / 8 are sampled; the sampled key nearest their mean is
//           the anchor when centring on it lowers the energy of the samples
//           without growing their range by more than 12.5 %, else -1.
//   Q/K     quant_int8_tile with ROTATE (fused.cu:202-407): v = x - x[anchor]
//           (K only), v = H v with H the sign-diagonal normalised
//           Walsh-Hadamard transform (attention_hadamard8, :206-260), then
//           per tile (Q 16 tokens, K 64 tokens) amax = max(1e-7, max |v|),
//           scale = amax / 127, q = cvt.rni.sat.s8(v * (127 / amax)).
//   V       quantize_value_kernel (quant_v_int8_cuda_sm75.cu:58-164):
//           scale[c] = max(amax_c / 127, 1e-12) over all tokens,
//           q = cvt.rni.sat.s8(v * (1 / scale[c])).
// Every reduction here is a max (exact in any order) except the anchor's
// energy sums, which keep the reference's order: one channel per thread,
// 32-lane trees, the four tree results added from 0 in order.
//
// MI355X layout of V: channel-major codes [B][H][D][Lpad] with keys in
// natural order (the INT8 PV MFMA reads 16 consecutive keys of one channel
// per lane).
#include <algorithm>
#include <type_traits>

#include "w8a8_common.h"

namespace tu {
namespace {

template <bool kFp16>
__device__ __forceinline__ float h_to_f32(uint32_t bits16) {
    if constexpr (kFp16) return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits16)));
    else return __uint_as_float(bits16 << 16);
}

// cvt.rni.sat.s8.f32 (round half to even, saturate to [-128, 127]) of four
// values packed little-endian, without conversions: the clamp comes first
// (the bounds are integers, so clamping and rounding commute; NaN clamps to
// -128), then adding 1.5 * 2^23 rounds half to even to an integer whose two's
// complement sits in the low byte.
__device__ __forceinline__ uint32_t sat_rne_s8x4(float a, float b, float c, float d) {
    const float vs[4] = {a, b, c, d};
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = __float_as_uint(fminf(127.0f, fmaxf(-128.0f, vs[k])) + 12582912.0f);
    // low bytes of two words, then of two pairs
    const uint32_t lo = __builtin_amdgcn_perm(w[1], w[0], 0x0c0c0400u);
    const uint32_t hi = __builtin_amdgcn_perm(w[3], w[2], 0x0c0c0400u);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// ---------------------------------------------------------------------------
// K anchor: one workgroup of 128 threads (two wave64 = four 32-lane trees)
// per (kv head, batch).
// ---------------------------------------------------------------------------
template <bool kFp16>
__device__ __forceinline__ void anchor_body(const uint16_t *__restrict__ k, int64_t len, int dim, int64_t s_b,
                                            int64_t s_h, int64_t s_l, int32_t *__restrict__ anchors, int64_t h,
                                            int64_t b, int64_t heads) {
    __shared__ float samples[kAnchorSamples][128];
    const int c = threadIdx.x;
    const uint16_t *kb = k + b * s_b + h * s_h;
#pragma unroll
    for (int s = 0; s < kAnchorSamples; ++s) {
        const int64_t row = static_cast<int64_t>(s) * (len - 1) / (kAnchorSamples - 1);
        samples[s][c] = c < dim ? h_to_f32<kFp16>(kb[row * s_l + c]) : 0.0f;
    }
    __syncthreads();
    const int sel = w8a8_anchor_decide(samples, dim);
    if (c == 0)
        anchors[b * heads + h] =
            sel >= 0 ? static_cast<int32_t>(static_cast<int64_t>(sel) * (len - 1) / (kAnchorSamples - 1)) : -1;
}

template <bool kFp16>
__global__ __launch_bounds__(kAnchorThreads) void anchor_kernel(const uint16_t *__restrict__ k, int64_t len, int dim,
                                                                int64_t s_b, int64_t s_h, int64_t s_l,
                                                                int32_t *__restrict__ anchors) {
    anchor_body<kFp16>(k, len, dim, s_b, s_h, s_l, anchors, blockIdx.x, blockIdx.y, gridDim.x);
}

// ---------------------------------------------------------------------------
// Rotated Q/K quantizer: one workgroup (4 wave64) per 64-token chunk of a
// head, Q heads first, then K heads.  A thread owns one pack of 8 channels
// of kIters tokens; the D / 8 packs of a token are consecutive lanes, so the
// transform's cross-pack butterfly is a lane xor.  A Q tile (16 tokens) is
// covered by whole wave-passes, so its amax is a wave max plus an exchange
// through LDS.
// ---------------------------------------------------------------------------
constexpr int kQkThreads = 256;
constexpr int kChunk = 64;

struct RotArgs {
    const uint16_t *x[2];
    int8_t *out[2];
    float *scale[2];
    const int32_t *anchors;  // [B][Hk] or null
    int64_t heads[2], len[2], ntiles[2];
    int64_t x_sb[2], x_sh[2], x_sl[2];
    int64_t o_sb[2], o_sh[2], o_sl[2];
    int rotate;
    int wide;  // head_dim 64 into 128-byte rows, channels 64 .. 127 zero
};

template <bool kFp16, int D>
__device__ __forceinline__ void rot_quant_body(const RotArgs &args, uint32_t task, int64_t b) {
    constexpr int kPacks = D / 8;
    constexpr int kTokPerPass = kQkThreads / kPacks;   // 16 (D 128) or 32 (D 64)
    constexpr int kIters = kChunk / kTokPerPass;        // 4 or 2
    constexpr int kWaveTok = 64 / kPacks;               // tokens of one wave-pass
    __shared__ float wave_amax[kIters][kQkThreads / 64];

    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int pack = tid % kPacks;
    // 32-bit block arithmetic: a 64-bit division is a long instruction sequence
    const uint32_t nq_blocks = static_cast<uint32_t>(args.heads[0]) * static_cast<uint32_t>(args.ntiles[0] / 4);
    const int which = task < nq_blocks ? 0 : 1;
    if (which) task -= nq_blocks;
    const int64_t len = args.len[which];
    const uint32_t nch = static_cast<uint32_t>((len + kChunk - 1) / kChunk);
    const int64_t head = task / nch;
    const int64_t chunk = task % nch;
    const int64_t t0 = chunk * kChunk;
    const uint16_t *xbase = args.x[which] + b * args.x_sb[which] + head * args.x_sh[which];

    float anchor[8];
    bool anchored = false;
    if (which == 1 && args.anchors != nullptr) {
        const int32_t a = args.anchors[b * args.heads[1] + head];
        anchored = a >= 0;
        if (anchored) {
            const u32x4 raw = *reinterpret_cast<const u32x4 *>(xbase + static_cast<int64_t>(a) * args.x_sl[1] + pack * 8);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                anchor[2 * j] = h_to_f32<kFp16>(raw[j] & 0xffffu);
                anchor[2 * j + 1] = h_to_f32<kFp16>(raw[j] >> 16);
            }
        }
    }

    float v[kIters][8];
    float amax[kIters];
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        const int64_t t = t0 + it * kTokPerPass + tid / kPacks;
        u32x4 raw = u32x4{0u, 0u, 0u, 0u};
        if (t < len) raw = *reinterpret_cast<const u32x4 *>(xbase + t * args.x_sl[which] + pack * 8);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[it][2 * j] = h_to_f32<kFp16>(raw[j] & 0xffffu);
            v[it][2 * j + 1] = h_to_f32<kFp16>(raw[j] >> 16);
        }
        if (anchored && t < len) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[it][j] = v[it][j] - anchor[j];
        }
        if (args.rotate) w8a8_hadamard_pack<D>(v[it], pack);
        float a = 0.0000001f;
#pragma unroll
        for (int j = 0; j < 8; ++j) a = fmaxf(a, fabsf(v[it][j]));
        amax[it] = wave_max_nonneg(a);   // a >= 1e-7 and never NaN (fmaxf passes NaN over)
    }
    if ((tid & 63) == 0) {
#pragma unroll
        for (int it = 0; it < kIters; ++it) wave_amax[it][wave] = amax[it];
    }
    __syncthreads();

    // Scale of each token's tile: Q tiles of 16 tokens, one K tile per chunk.
    float mult[kIters];
    if (which == 0) {
        // Q tile s = tokens [16 s, 16 s + 16) of the chunk: the max of the
        // wave-passes inside it.
        constexpr int kSubs = kChunk / 16;
        float sub_amax[kSubs];
#pragma unroll
        for (int s = 0; s < kSubs; ++s) sub_amax[s] = 0.0f;
#pragma unroll
        for (int w = 0; w < kQkThreads / 64; ++w)
#pragma unroll
            for (int i2 = 0; i2 < kIters; ++i2) {
                const int s = (i2 * kTokPerPass + w * kWaveTok) / 16;
                sub_amax[s] = fmaxf(sub_amax[s], wave_amax[i2][w]);
            }
#pragma unroll
        for (int it = 0; it < kIters; ++it) {
            const int mine = (it * kTokPerPass + wave * kWaveTok) / 16;
            float a = sub_amax[0];
#pragma unroll
            for (int s = 1; s < kSubs; ++s) a = mine == s ? sub_amax[s] : a;
            mult[it] = 127.0f / a;
        }
        if (tid < kSubs) {
            float a = sub_amax[0];
#pragma unroll
            for (int s = 1; s < kSubs; ++s) a = tid == s ? sub_amax[s] : a;
            args.scale[0][(b * args.heads[0] + head) * args.ntiles[0] + chunk * kSubs + tid] = a / 127.0f;
        }
    } else {
        float a = 0.0f;
#pragma unroll
        for (int w = 0; w < kQkThreads / 64; ++w)
#pragma unroll
            for (int i2 = 0; i2 < kIters; ++i2) a = fmaxf(a, wave_amax[i2][w]);
#pragma unroll
        for (int it = 0; it < kIters; ++it) mult[it] = 127.0f / a;
        if (tid == 0) args.scale[1][(b * args.heads[1] + head) * args.ntiles[1] + chunk] = a / 127.0f;
    }

    int8_t *obase = args.out[which] + b * args.o_sb[which] + head * args.o_sh[which];
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        const int64_t t = t0 + it * kTokPerPass + tid / kPacks;
        if (t >= len) continue;
        float y[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = v[it][j] * mult[it];
        const u32x2 packed{sat_rne_s8x4(y[0], y[1], y[2], y[3]), sat_rne_s8x4(y[4], y[5], y[6], y[7])};
        int8_t *dst = obase + t * args.o_sl[which] + pack * 8;
        *reinterpret_cast<u32x2 *>(dst) = packed;
        if (D == 64 && args.wide) *reinterpret_cast<u32x2 *>(dst + 64) = u32x2{0u, 0u};
    }
}

template <bool kFp16, int D>
__global__ __launch_bounds__(kQkThreads) void rot_quant_kernel(RotArgs args) {
    rot_quant_body<kFp16, D>(args, blockIdx.x, blockIdx.y);
}

// ---------------------------------------------------------------------------
// V: per-channel amax over token chunks, then codes.  Every code workgroup
// reduces its head's chunk maxima itself (at most 64 rows of 512 bytes from
// L2): a launch for the scales alone costs more than that.
// ---------------------------------------------------------------------------
constexpr int kVThreads = 256;
constexpr int kAmaxThreads = kAnchorThreads;
constexpr int64_t kAmaxTokens = 128;  // fewest tokens of an amax chunk

// Tokens of an amax chunk: 128, more where that would pass 64 chunks a head,
// or 16 once the heads alone fill the GPU.
int64_t v_chunk_tokens(int64_t bh, int64_t len) {
    const int64_t most = std::max<int64_t>(16, std::min<int64_t>(64, 1024 / bh));
    const int64_t chunks = std::min<int64_t>((len + kAmaxTokens - 1) / kAmaxTokens, most);
    return (len + chunks - 1) / chunks;
}
int64_t v_chunks(int64_t bh, int64_t len) {
    const int64_t tokens = v_chunk_tokens(bh, len);
    return (len + tokens - 1) / tokens;
}

struct VArgs {
    const uint16_t *v;
    int64_t heads, len, lpad, s_b, s_h, s_l;
    int64_t chunk_tokens, chunks;
    float *partial;  // [B][H][chunks][D]
    float *scale;    // [B][H][D], or [B][H][128] when wide
    int8_t *vq;      // channel-major codes, D or (wide) 128 channels
    int wide;
};

template <bool kFp16, int D>
__device__ __forceinline__ void v_amax_body(const VArgs &a, int64_t chunk, int64_t h, int64_t b) {
    constexpr int kPacks = D / 8;
    constexpr int kRows = kAmaxThreads / kPacks;
    __shared__ float wave_max[kAmaxThreads / 64][D];
    const int tid = threadIdx.x;
    const int pack = tid % kPacks;
    const uint16_t *base = a.v + b * a.s_b + h * a.s_h;
    float m[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = 0.0f;
    const int64_t t_end = min(a.len, (chunk + 1) * a.chunk_tokens);
#pragma unroll 8
    for (int64_t t = chunk * a.chunk_tokens + tid / kPacks; t < t_end; t += kRows) {
        const u32x4 raw = *reinterpret_cast<const u32x4 *>(base + t * a.s_l + pack * 8);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            m[2 * j] = fmaxf(m[2 * j], fabsf(h_to_f32<kFp16>(raw[j] & 0xffffu)));
            m[2 * j + 1] = fmaxf(m[2 * j + 1], fabsf(h_to_f32<kFp16>(raw[j] >> 16)));
        }
    }
    // lanes l, l + kPacks, ... of a wave hold the same channels
#pragma unroll
    for (int off = kPacks; off < 64; off <<= 1)
#pragma unroll
        for (int j = 0; j < 8; ++j) m[j] = fmaxf(m[j], __shfl_xor(m[j], off));
    if ((tid & 63) < kPacks) {
#pragma unroll
        for (int j = 0; j < 8; ++j) wave_max[tid >> 6][pack * 8 + j] = m[j];
    }
    __syncthreads();
    if (tid < D) {
        float x = 0.0f;
#pragma unroll
        for (int w = 0; w < kAmaxThreads / 64; ++w) x = fmaxf(x, wave_max[w][tid]);
        a.partial[((b * a.heads + h) * a.chunks + chunk) * D + tid] = x;
    }
}

// One workgroup per 64-key tile: codes through an LDS byte tile (rows of D
// + 16 bytes), written channel-major as 16-byte key runs.
template <bool kFp16, int D>
__device__ __forceinline__ void v_quant_body(const VArgs &a, int64_t tix, int64_t h, int64_t b) {
    constexpr int kPacks = D / 8;
    constexpr int kRows = kVThreads / kPacks;
    constexpr int kIters = 64 / kRows;
    constexpr int kRowBytes = D + 16;
    constexpr int kParts = kVThreads / D;  // threads that share a channel's chunks
    __shared__ __align__(16) int8_t tile[64 * kRowBytes];
    __shared__ float part_max[kParts][D];
    __shared__ __align__(16) float inv_scale[D];
    const int tid = threadIdx.x;
    const int pack = tid % kPacks;
    const int64_t bh = b * a.heads + h;
    const int64_t dout = a.wide ? 128 : D;
    const uint16_t *base = a.v + b * a.s_b + h * a.s_h;
    u32x4 raw[kIters];
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        const int64_t t = tix * 64 + it * kRows + tid / kPacks;
        raw[it] = u32x4{0u, 0u, 0u, 0u};
        if (t < a.len) raw[it] = *reinterpret_cast<const u32x4 *>(base + t * a.s_l + pack * 8);
    }
    float m = 0.0f;
#pragma unroll 4
    for (int64_t i = tid / D; i < a.chunks; i += kParts) m = fmaxf(m, a.partial[(bh * a.chunks + i) * D + tid % D]);
    part_max[tid / D][tid % D] = m;
    __syncthreads();
    if (tid < D) {
#pragma unroll
        for (int i = 0; i < kParts; ++i) m = fmaxf(m, part_max[i][tid]);
        const float scale = fmaxf(m / 127.0f, 1.0e-12f);
        inv_scale[tid] = 1.0f / scale;
        if (tix == 0) {
            a.scale[bh * dout + tid] = scale;
            if (a.wide) a.scale[bh * dout + 64 + tid] = 1.0e-12f;  // D = 64
        }
    }
    __syncthreads();
    float inv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) inv[j] = inv_scale[pack * 8 + j];
#pragma unroll
    for (int it = 0; it < kIters; ++it) {
        float y[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            y[2 * j] = h_to_f32<kFp16>(raw[it][j] & 0xffffu) * inv[2 * j];
            y[2 * j + 1] = h_to_f32<kFp16>(raw[it][j] >> 16) * inv[2 * j + 1];
        }
        *reinterpret_cast<u32x2 *>(tile + (it * kRows + tid / kPacks) * kRowBytes + pack * 8) =
            u32x2{sat_rne_s8x4(y[0], y[1], y[2], y[3]), sat_rne_s8x4(y[4], y[5], y[6], y[7])};
    }
    __syncthreads();
    // item = (channel, 16-key run)
#pragma unroll
    for (int item = tid; item < D * 4; item += kVThreads) {
        const int c = item >> 2, run = item & 3;
        u32x4 out;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            uint32_t word = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int8_t code = tile[(run * 16 + 4 * w + e) * kRowBytes + c];
                word |= (static_cast<uint32_t>(code) & 0xffu) << (8 * e);
            }
            out[w] = word;
        }
        int8_t *dst = a.vq + (bh * dout + c) * a.lpad + tix * 64 + run * 16;
        *reinterpret_cast<u32x4 *>(dst) = out;
        if (D == 64 && a.wide) *reinterpret_cast<u32x4 *>(dst + 64 * a.lpad) = u32x4{0u, 0u, 0u, 0u};
    }
}

template <bool kFp16, int D>
__global__ __launch_bounds__(kAmaxThreads) void v_amax_kernel(VArgs a) {
    v_amax_body<kFp16, D>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <bool kFp16, int D>
__global__ __launch_bounds__(kVThreads) void v_quant_kernel(VArgs a) {
    v_quant_body<kFp16, D>(a, blockIdx.x, blockIdx.y, blockIdx.z);
}

// ---------------------------------------------------------------------------
// The whole prologue in two launches (five kernels one after the other left
// most of the GPU idle on ordinary lengths): what needs only the inputs, the
// K anchors and the V chunk maxima, then what needs those, the Q / K and the
// V codes.  Workgroups in that order along x, batches along y.
// ---------------------------------------------------------------------------
template <bool kFp16, int D>
__global__ __launch_bounds__(kAnchorThreads) void w8a8_prep_stats_kernel(RotArgs r, VArgs a, int32_t *anchors,
                                                                         uint32_t anchor_blocks) {
    const uint32_t id = blockIdx.x, chunks = static_cast<uint32_t>(a.chunks);
    const int64_t b = blockIdx.y;
    if (id < anchor_blocks)
        anchor_body<kFp16>(r.x[1], r.len[1], D, r.x_sb[1], r.x_sh[1], r.x_sl[1], anchors, id, b, r.heads[1]);
    else
        v_amax_body<kFp16, D>(a, (id - anchor_blocks) % chunks, (id - anchor_blocks) / chunks, b);
}

template <bool kFp16, int D>
__global__ __launch_bounds__(kVThreads) void w8a8_prep_codes_kernel(RotArgs r, VArgs a, uint32_t rot_blocks) {
    const uint32_t id = blockIdx.x, tiles = static_cast<uint32_t>(a.lpad / 64);
    const int64_t b = blockIdx.y;
    if (id < rot_blocks) rot_quant_body<kFp16, D>(r, id, b);
    else v_quant_body<kFp16, D>(a, (id - rot_blocks) % tiles, (id - rot_blocks) / tiles, b);
}

// Argument checks and kernel arguments shared by the entry points (host only).
int32_t check_qk(const void *q, const void *k, int32_t dtype, int64_t batch, int64_t hq, int64_t hk, int64_t lq,
                 int64_t lk, int64_t dim, int64_t q_sb, int64_t q_sh, int64_t q_sl, int64_t k_sb, int64_t k_sh,
                 int64_t k_sl, int8_t *q8, int64_t q8_sb, int64_t q8_sh, int64_t q8_sl, int8_t *k8, int64_t k8_sb,
                 int64_t k8_sh, int64_t k8_sl, float *q_scale, float *k_scale) {
    TU_REQUIRE(dtype == 0 || dtype == 1, "W8A8 Q/K dtype must be 0 (bf16) or 1 (fp16)");
    TU_REQUIRE(dim == 64 || dim == 128, "W8A8 Q/K quantizer requires head_dim 64 or 128, got %lld",
               static_cast<long long>(dim));
    TU_REQUIRE(batch > 0 && hq > 0 && hk > 0 && lq > 0 && lk > 0 && batch <= 65535,
               "W8A8 Q/K quantizer dimensions out of range");
    TU_REQUIRE(q && k && q8 && k8 && q_scale && k_scale, "W8A8 Q/K quantizer pointers must be non-null");
    const int64_t nq = (lq + kChunk - 1) / kChunk, nk = (lk + kChunk - 1) / kChunk;
    TU_REQUIRE(hq * nq + hk * nk <= 0x7fffffff, "W8A8 Q/K quantizer grid too large");
    TU_REQUIRE(q_sb % 8 == 0 && q_sh % 8 == 0 && q_sl % 8 == 0 && k_sb % 8 == 0 && k_sh % 8 == 0 && k_sl % 8 == 0 &&
                   (reinterpret_cast<uintptr_t>(q) & 15) == 0 && (reinterpret_cast<uintptr_t>(k) & 15) == 0,
               "W8A8 Q/K inputs need 16-byte aligned rows");
    TU_REQUIRE(q8_sb % 8 == 0 && q8_sh % 8 == 0 && q8_sl % 8 == 0 && k8_sb % 8 == 0 && k8_sh % 8 == 0 &&
                   k8_sl % 8 == 0 && (reinterpret_cast<uintptr_t>(q8) & 7) == 0 &&
                   (reinterpret_cast<uintptr_t>(k8) & 7) == 0,
               "W8A8 Q/K codes need 8-byte aligned rows");
    return 0;
}

RotArgs rot_args(const void *q, const void *k, int64_t hq, int64_t hk, int64_t lq, int64_t lk, int64_t q_sb,
                 int64_t q_sh, int64_t q_sl, int64_t k_sb, int64_t k_sh, int64_t k_sl, int8_t *q8, int64_t q8_sb,
                 int64_t q8_sh, int64_t q8_sl, int8_t *k8, int64_t k8_sb, int64_t k8_sh, int64_t k8_sl, float *q_scale,
                 float *k_scale, const int32_t *anchors, int32_t rotate) {
    const int64_t nq = (lq + kChunk - 1) / kChunk, nk = (lk + kChunk - 1) / kChunk;
    RotArgs a{};
    a.x[0] = static_cast<const uint16_t *>(q);
    a.x[1] = static_cast<const uint16_t *>(k);
    a.out[0] = q8;
    a.out[1] = k8;
    a.scale[0] = q_scale;
    a.scale[1] = k_scale;
    a.anchors = anchors;
    a.heads[0] = hq;
    a.heads[1] = hk;
    a.len[0] = lq;
    a.len[1] = lk;
    a.ntiles[0] = nq * 4;
    a.ntiles[1] = nk;
    a.x_sb[0] = q_sb; a.x_sh[0] = q_sh; a.x_sl[0] = q_sl;
    a.x_sb[1] = k_sb; a.x_sh[1] = k_sh; a.x_sl[1] = k_sl;
    a.o_sb[0] = q8_sb; a.o_sh[0] = q8_sh; a.o_sl[0] = q8_sl;
    a.o_sb[1] = k8_sb; a.o_sh[1] = k8_sh; a.o_sl[1] = k8_sl;
    a.rotate = rotate != 0;
    return a;
}

int32_t check_v(const void *v, int32_t dtype, int64_t batch, int64_t heads, int64_t len, int64_t dim, int64_t s_b,
                int64_t s_h, int64_t s_l, int8_t *vq, int64_t lpad, float *scale, void *workspace,
                int64_t workspace_bytes) {
    TU_REQUIRE(dtype == 0 || dtype == 1, "W8A8 V dtype must be 0 (bf16) or 1 (fp16)");
    TU_REQUIRE(dim == 64 || dim == 128, "W8A8 V quantizer requires head_dim 64 or 128, got %lld",
               static_cast<long long>(dim));
    TU_REQUIRE(batch > 0 && heads > 0 && len > 0 && batch <= 65535 && heads <= 65535,
               "W8A8 V quantizer dimensions out of range");
    TU_REQUIRE(lpad == (len + 63) / 64 * 64, "W8A8 V padded length must be ceil(len / 64) * 64");
    TU_REQUIRE(v && vq && scale && workspace, "W8A8 V quantizer pointers must be non-null");
    TU_REQUIRE(workspace_bytes >= batch * heads * dim * v_chunks(batch * heads, len) * 4,
               "W8A8 V quantizer workspace too small");
    TU_REQUIRE(s_b % 8 == 0 && s_h % 8 == 0 && s_l % 8 == 0 && (reinterpret_cast<uintptr_t>(v) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(vq) & 15) == 0 && (reinterpret_cast<uintptr_t>(workspace) & 3) == 0,
               "W8A8 V quantizer needs 16-byte aligned rows");
    return 0;
}

VArgs v_args(const void *v, int64_t batch, int64_t heads, int64_t len, int64_t s_b, int64_t s_h, int64_t s_l,
             int8_t *vq, int64_t lpad, float *scale, void *workspace, int wide) {
    return VArgs{static_cast<const uint16_t *>(v), heads, len, lpad, s_b, s_h, s_l,
                 v_chunk_tokens(batch * heads, len), v_chunks(batch * heads, len),
                 static_cast<float *>(workspace), scale, vq, wide};
}

// f(kFp16, D) as compile-time constants.
template <typename F>
void with_type_and_dim(int32_t dtype, int64_t dim, F &&f) {
    using std::bool_constant;
    using std::integral_constant;
    if (dtype) {
        if (dim == 128) f(bool_constant<true>{}, integral_constant<int, 128>{});
        else f(bool_constant<true>{}, integral_constant<int, 64>{});
    } else {
        if (dim == 128) f(bool_constant<false>{}, integral_constant<int, 128>{});
        else f(bool_constant<false>{}, integral_constant<int, 64>{});
    }
}

}  // namespace
}  // namespace tu

extern "C" int32_t tu_w8a8_quant_qk(const void *q, const void *k, int32_t dtype, int64_t batch, int64_t hq,
                                    int64_t hk, int64_t lq, int64_t lk, int64_t dim, int64_t q_sb, int64_t q_sh,
                                    int64_t q_sl, int64_t k_sb, int64_t k_sh, int64_t k_sl, int8_t *q8,
                                    int64_t q8_sb, int64_t q8_sh, int64_t q8_sl, int8_t *k8, int64_t k8_sb,
                                    int64_t k8_sh, int64_t k8_sl, float *q_scale, float *k_scale,
                                    int32_t *anchors, int32_t rotate, void *stream) {
    using namespace tu;
    if (check_qk(q, k, dtype, batch, hq, hk, lq, lk, dim, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, q8, q8_sb, q8_sh, q8_sl,
                 k8, k8_sb, k8_sh, k8_sl, q_scale, k_scale))
        return -1;
    if (require_gfx950()) return -1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const RotArgs a = rot_args(q, k, hq, hk, lq, lk, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, q8, q8_sb, q8_sh, q8_sl, k8,
                               k8_sb, k8_sh, k8_sl, q_scale, k_scale, anchors, rotate);
    const dim3 grid(static_cast<unsigned>(hq * (a.ntiles[0] / 4) + hk * a.ntiles[1]), static_cast<unsigned>(batch));
    const dim3 heads(static_cast<unsigned>(hk), static_cast<unsigned>(batch));
    with_type_and_dim(dtype, dim, [&](auto f16, auto d) {
        if (anchors != nullptr)
            anchor_kernel<f16.value><<<heads, kAnchorThreads, 0, s>>>(a.x[1], lk, static_cast<int>(dim), k_sb, k_sh,
                                                                      k_sl, anchors);
        rot_quant_kernel<f16.value, d.value><<<grid, kQkThreads, 0, s>>>(a);
    });
    return check_launch("tu_w8a8_quant_qk");
}

extern "C" int64_t tu_w8a8_quant_v_workspace(int64_t batch, int64_t heads, int64_t len, int64_t dim) {
    if (batch <= 0 || heads <= 0 || len <= 0 || dim <= 0) return -1;
    // chunk maxima (fp32)
    return batch * heads * dim * tu::v_chunks(batch * heads, len) * 4;
}

extern "C" int32_t tu_w8a8_quant_v(const void *v, int32_t dtype, int64_t batch, int64_t heads, int64_t len,
                                   int64_t dim, int64_t s_b, int64_t s_h, int64_t s_l, int8_t *vq, int64_t lpad,
                                   float *scale, void *workspace, int64_t workspace_bytes,
                                   void *stream) {
    using namespace tu;
    if (check_v(v, dtype, batch, heads, len, dim, s_b, s_h, s_l, vq, lpad, scale, workspace, workspace_bytes)) return -1;
    if (require_gfx950()) return -1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const VArgs a = v_args(v, batch, heads, len, s_b, s_h, s_l, vq, lpad, scale, workspace, 0);
    const unsigned h = static_cast<unsigned>(heads), b = static_cast<unsigned>(batch);
    with_type_and_dim(dtype, dim, [&](auto f16, auto d) {
        v_amax_kernel<f16.value, d.value><<<dim3(static_cast<unsigned>(a.chunks), h, b), kAmaxThreads, 0, s>>>(a);
        v_quant_kernel<f16.value, d.value><<<dim3(static_cast<unsigned>(lpad / 64), h, b), kVThreads, 0, s>>>(a);
    });
    return check_launch("tu_w8a8_quant_v");
}

extern "C" int32_t tu_w8a8_prep(const void *q, const void *k, const void *v, int32_t dtype, int64_t batch, int64_t hq,
                                int64_t hk, int64_t lq, int64_t lk, int64_t dim, int64_t q_sb, int64_t q_sh,
                                int64_t q_sl, int64_t k_sb, int64_t k_sh, int64_t k_sl, int64_t v_sb, int64_t v_sh,
                                int64_t v_sl, int8_t *q8, int64_t q8_sb, int64_t q8_sh, int64_t q8_sl, int8_t *k8,
                                int64_t k8_sb, int64_t k8_sh, int64_t k8_sl, float *q_scale, float *k_scale,
                                int32_t *anchors, int32_t rotate, int8_t *vq, int64_t lpad, float *v_scale,
                                int32_t wide, void *workspace, int64_t workspace_bytes, void *stream) {
    using namespace tu;
    if (check_qk(q, k, dtype, batch, hq, hk, lq, lk, dim, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, q8, q8_sb, q8_sh, q8_sl,
                 k8, k8_sb, k8_sh, k8_sl, q_scale, k_scale))
        return -1;
    if (check_v(v, dtype, batch, hk, lk, dim, v_sb, v_sh, v_sl, vq, lpad, v_scale, workspace, workspace_bytes)) return -1;
    TU_REQUIRE(!wide || (dim == 64 && q8_sl >= 128 && k8_sl >= 128), "W8A8 wide codes are for head_dim 64 in rows of 128");
    RotArgs r = rot_args(q, k, hq, hk, lq, lk, q_sb, q_sh, q_sl, k_sb, k_sh, k_sl, q8, q8_sb, q8_sh, q8_sl, k8, k8_sb,
                         k8_sh, k8_sl, q_scale, k_scale, anchors, rotate);
    r.wide = wide != 0;
    const VArgs a = v_args(v, batch, hk, lk, v_sb, v_sh, v_sl, vq, lpad, v_scale, workspace, r.wide);
    const int64_t anchor_blocks = anchors != nullptr ? hk : 0;
    const int64_t rot_blocks = hq * (r.ntiles[0] / 4) + hk * r.ntiles[1];
    const int64_t stats = anchor_blocks + hk * a.chunks, codes = rot_blocks + hk * (lpad / 64);
    TU_REQUIRE(stats <= 0x7fffffff && codes <= 0x7fffffff, "W8A8 prologue grid too large");
    if (require_gfx950()) return -1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const unsigned b = static_cast<unsigned>(batch);
    with_type_and_dim(dtype, dim, [&](auto f16, auto d) {
        w8a8_prep_stats_kernel<f16.value, d.value>
            <<<dim3(static_cast<unsigned>(stats), b), kAnchorThreads, 0, s>>>(r, a, anchors, static_cast<uint32_t>(anchor_blocks));
        w8a8_prep_codes_kernel<f16.value, d.value>
            <<<dim3(static_cast<unsigned>(codes), b), kVThreads, 0, s>>>(r, a, static_cast<uint32_t>(rot_blocks));
    });
    return check_launch("tu_w8a8_prep");
}
