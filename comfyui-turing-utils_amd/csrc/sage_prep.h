// Device bodies of the Sage prologue: K chunk sums, per-block INT8
// quantization and the V transpose, each for one workgroup of 256 threads at
// a given (block, head, batch), shared by their own kernels and the fused
// prologue (sage_quant.hip).
#pragma once

#include "tu_common.h"

namespace tu {

constexpr int kPrepThreads = 256;
constexpr int kPrepKeys = 64;  // keys of a V^T tile

// Sum over the 128 tokens of a chunk; partial: LDS [kPrepThreads / (D / 8)][D].
template <int D>
__device__ __forceinline__ void kmean_chunk(const uint16_t *__restrict__ k, int64_t len, int64_t s_b, int64_t s_h,
                                            int64_t s_l, float *__restrict__ chunk_sums, int64_t chunk, int64_t h,
                                            int64_t b, int64_t heads, int64_t chunks, float (*partial)[D]) {
    constexpr int kLanesPerRow = D / 8;
    constexpr int kRows = kPrepThreads / kLanesPerRow;
    constexpr int kPer = 128 / kRows;

    const int tid = threadIdx.x;
    const int r = tid / kLanesPerRow;
    const int c8 = tid % kLanesPerRow;
    const uint16_t *base = k + b * s_b + h * s_h;

    float s[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e] = 0.0f;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int64_t t = chunk * 128 + r + static_cast<int64_t>(kRows) * j;
        if (t < len) {
            const u32x4 v = *reinterpret_cast<const u32x4 *>(base + t * s_l + c8 * 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[2 * e] = s[2 * e] + bf16_bits_to_f32(v[e] & 0xffffu);
                s[2 * e + 1] = s[2 * e + 1] + bf16_bits_to_f32(v[e] >> 16);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) partial[r][c8 * 8 + e] = s[e];
    __syncthreads();
    if (tid < D) {
        float acc = 0.0f;
#pragma unroll 8
        for (int rr = 0; rr < kRows; ++rr) acc = acc + partial[rr][tid];
        chunk_sums[((b * heads + h) * chunks + chunk) * D + tid] = acc;
    }
}

__device__ __forceinline__ int32_t sat_rne_s8(float v) {
    if (v != v) return 0;
    const float r = fminf(127.0f, fmaxf(-128.0f, __builtin_rintf(v)));
    return static_cast<int32_t>(r);
}

// One workgroup per (token block, head, batch).  Each thread owns 8
// contiguous channels of every (256 / (D/8))-th token row of the block; the
// block is held in registers between the absmax and the quantization pass.
// mean_of(mu, c8) fills the means of channels 8 c8 .. 8 c8 + 7; wave_amax: LDS
// [kPrepThreads / 64].
template <int D, int BLK, bool kSubMean, typename Mean>
__device__ __forceinline__ void quant_block(
    const uint16_t *__restrict__ x, Mean mean_of, int64_t len, int64_t s_b, int64_t s_h, int64_t s_l,
    int8_t *__restrict__ q, int64_t q_b, int64_t q_h, int64_t q_l, float *__restrict__ scale, int64_t blk, int64_t h,
    int64_t b, int64_t heads, int64_t nblk, float *wave_amax) {
    constexpr int kLanesPerRow = D / 8;
    constexpr int kRowsPerPass = kPrepThreads / kLanesPerRow;
    constexpr int kPasses = (BLK + kRowsPerPass - 1) / kRowsPerPass;

    const int tid = threadIdx.x;
    const int r = tid / kLanesPerRow;
    const int c8 = tid % kLanesPerRow;
    const uint16_t *xb = x + b * s_b + h * s_h;
    int8_t *qb = q + b * q_b + h * q_h;

    float mu[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) mu[e] = 0.0f;
    if constexpr (kSubMean) mean_of(mu, c8);

    float v[kPasses][8];
    float amax = 0.0000001f;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const int row = r + p * kRowsPerPass;
        const int64_t t = blk * BLK + row;
        if (row < BLK && t < len) {
            const u32x4 xv = *reinterpret_cast<const u32x4 *>(xb + t * s_l + c8 * 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[p][2 * e] = bf16_bits_to_f32(xv[e] & 0xffffu);
                v[p][2 * e + 1] = bf16_bits_to_f32(xv[e] >> 16);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if constexpr (kSubMean) v[p][e] = v[p][e] - mu[e];
                amax = fmaxf(amax, fabsf(v[p][e]));
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[p][e] = 0.0f;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 64));
    if ((tid & 63) == 0) wave_amax[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(wave_amax[0], wave_amax[1]), fmaxf(wave_amax[2], wave_amax[3]));
    if (tid == 0) scale[(b * heads + h) * nblk + blk] = amax / 127.0f;
    const float mult = 127.0f / amax;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const int row = r + p * kRowsPerPass;
        const int64_t t = blk * BLK + row;
        if (row < BLK && t < len) {
            u32x2 out;
            uint32_t w[2];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                uint32_t acc = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc |= (static_cast<uint32_t>(sat_rne_s8(v[p][4 * hh + e] * mult)) & 0xffu) << (8 * e);
                w[hh] = acc;
            }
            out.x = w[0];
            out.y = w[1];
            *reinterpret_cast<u32x2 *>(qb + t * q_l + c8 * 8) = out;
        }
    }
}

// V [key][d] (bf16, strides) -> V^T [b][h][d][lpad] with zero keys in [lk, lpad).
// One workgroup per 64-key tile: 64 x 128 staged through LDS (rows padded to
// 132 elements so the column reads are bank-conflict free).
template <int D>
__device__ __forceinline__ void v_prep_tile(const uint16_t *__restrict__ v, int64_t lk, int64_t lpad, int64_t v_sb,
                                            int64_t v_sh, int64_t v_sl, uint16_t *__restrict__ vt, int64_t tile_i,
                                            int64_t h, int64_t b, int64_t heads, uint16_t (*tile)[D + 4]) {
    constexpr int kChunks = D / 8;             // 16-byte chunks of a key row
    constexpr int kRowsPerPass = 256 / kChunks;
    const int tid = threadIdx.x;
    const int64_t key0 = tile_i * kPrepKeys;
    const uint16_t *vp = v + b * v_sb + h * v_sh;
#pragma unroll
    for (int i = 0; i < kPrepKeys / kRowsPerPass; ++i) {
        const int row = i * kRowsPerPass + tid / kChunks;
        const int c = tid % kChunks;
        u32x4 val = u32x4{0u, 0u, 0u, 0u};
        if (key0 + row < lk) val = *reinterpret_cast<const u32x4 *>(vp + (key0 + row) * v_sl + c * 8);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            tile[row][c * 8 + 2 * e] = static_cast<uint16_t>(val[e] & 0xffffu);
            tile[row][c * 8 + 2 * e + 1] = static_cast<uint16_t>(val[e] >> 16);
        }
    }
    __syncthreads();
    uint16_t *dst = vt + (b * heads + h) * D * lpad + key0;
#pragma unroll
    for (int i = 0; i < D * 8 / 256; ++i) {
        const int item = tid + 256 * i;  // (d, 8-key chunk)
        const int d = item >> 3, c = item & 7;
        u32x4 out;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            out[e] = static_cast<uint32_t>(tile[c * 8 + 2 * e][d]) | (static_cast<uint32_t>(tile[c * 8 + 2 * e + 1][d]) << 16);
        *reinterpret_cast<u32x4 *>(dst + d * lpad + c * 8) = out;
    }
}

}  // namespace tu
