// The numbering of the attention kernels' workgroups, for the kernels and (in
// plain C++) for a test on the host.
#pragma once

#include <algorithm>
#include <cstdint>

#ifdef __HIPCC__
#define TU_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define TU_HOST_DEVICE inline
#endif

namespace tu {

// Workgroup i of n (XCD i mod 8) -> its place in the plan: XCD x owns the
// contiguous x-th eighth of the n, so the query blocks of a head run on one
// XCD and its L2 reads that head's K and V^T once for all of them.
TU_HOST_DEVICE uint32_t xcd_chunk(uint32_t i, uint32_t n) {
    const uint32_t x = i & 7, q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + (i >> 3);
}

// Work plan of a Sage launch.  Query blocks are numbered head-major (block =
// (batch * hq + head) * nqb + query block).  Non-causal: blocks below
// split_from run whole, one workgroup each; every later block runs as
// `parts` workgroups of seg_tiles key tiles (the last range may be shorter),
// all blocks' first ranges before any second range.  Causal: every block
// runs as ceil(its key tiles / seg_tiles) workgroups; workgroups are numbered
// by query block from the last, longest one to the first (heads fastest,
// then ranges), so the long ones start first and the short ones fill the
// end: at B2 H16 L4001 D128 that took the kernel from 177 to 115 us.
struct AttnPlan {
    uint32_t nqb;         // query blocks of a head
    uint32_t bh;          // batch * hq
    uint32_t split_from;  // first split block (non-causal)
    uint32_t parts;       // key ranges of a split block (causal: of the last query block)
    int seg_tiles;        // key tiles of a range
    int64_t part_row0;    // query row (batch * hq * lq numbering) of the first split block
    int64_t part_rows;    // query rows of the split blocks
};

struct SagePlace {
    uint32_t bh, qb, z;  // batch * head, query block, key range
    bool whole;          // its block runs as one workgroup (causal: left to the kernel, which knows the tiles)
};

template <bool kCausal, bool kSplit>
TU_HOST_DEVICE SagePlace sage_place(const AttnPlan &plan, uint32_t id) {
    SagePlace p{0, 0, 0, true};
    if constexpr (kCausal) {
        p.bh = id % plan.bh;
        id /= plan.bh;
        if constexpr (kSplit) {
            p.z = id % plan.parts;
            id /= plan.parts;
        }
        p.qb = plan.nqb - 1 - id;
    } else {
        const uint32_t blocks = plan.nqb * plan.bh;
        if (kSplit && id >= plan.split_from) {
            // Split blocks keep their order: the ranges of a launch that is
            // split are short, and 16 or more blocks of a head on one XCD
            // would all read the same key tile at once (B1 H4 L4001 D128,
            // four ranges: 39.1 us spread over the XCDs, 41.0 with a head's
            // on one; B1 H6 L3000 D64 27.5 and 31.4).
            const uint32_t n = blocks - plan.split_from;
            const uint32_t i = id - plan.split_from;
            p.z = i / n;
            id = plan.split_from + i - p.z * n;
            p.whole = false;
        } else {
            id = xcd_chunk(id, kSplit ? plan.split_from : blocks);
        }
        p.bh = id / plan.nqb;
        p.qb = id % plan.nqb;
    }
    return p;
}

// Workgroups of a launch.
template <bool kCausal>
inline int64_t sage_grid(const AttnPlan &plan) {
    const int64_t blocks = static_cast<int64_t>(plan.nqb) * plan.bh;
    if (plan.parts <= 1) return blocks;
    return kCausal ? blocks * plan.parts : plan.split_from + (blocks - plan.split_from) * plan.parts;
}

// Work plan of a W8A8 launch.  Query blocks of 256 rows are numbered head-major.
// Blocks below split_from run whole, one workgroup of 32 rows a wave; every
// later one as two workgroups of 128 rows, 16 a wave (an end block of at most
// 128 rows leaves its second one empty).  Neither changes a row's arithmetic.
// Causal workgroups are numbered by query block from the last, longest one
// to the first, heads fastest.
struct W8Plan {
    uint32_t nqb;         // query blocks of a head
    uint32_t bh;          // batch * hq
    uint32_t split_from;  // first block that runs as two workgroups (causal: all or none)
};

struct W8Place {
    uint32_t bh, qb, half;  // batch * head, query block, its first or second 128 rows
    bool whole;             // all 256 rows
};

// kMode: 0 every block whole, 1 every block in two, 2 both.
template <bool kCausal, int kMode>
TU_HOST_DEVICE W8Place w8_place(const W8Plan &plan, uint32_t id) {
    W8Place p{0, 0, 0, kMode == 0};
    if constexpr (kCausal) {
        p.bh = id % plan.bh;
        id /= plan.bh;
        if constexpr (kMode == 1) {
            p.half = 1 - (id & 1);  // the later rows are the longer ones
            id >>= 1;
        }
        p.qb = plan.nqb - 1 - id;
    } else {
        const uint32_t blocks = plan.nqb * plan.bh;
        if constexpr (kMode == 2) p.whole = id < plan.split_from;
        if (p.whole) {
            id = xcd_chunk(id, kMode == 0 ? blocks : plan.split_from);
        } else {
            const uint32_t from = kMode == 1 ? 0 : plan.split_from;
            id = xcd_chunk(id - from, 2 * (blocks - from));
            p.half = id & 1;
            id = from + (id >> 1);
        }
        p.bh = id / plan.nqb;
        p.qb = id % plan.nqb;
    }
    return p;
}

// Workgroups of a launch.
inline int64_t w8_grid(const W8Plan &plan) {
    const int64_t blocks = static_cast<int64_t>(plan.nqb) * plan.bh;
    const int64_t whole = std::min<int64_t>(plan.split_from, blocks);
    return whole + 2 * (blocks - whole);
}

}  // namespace tu
