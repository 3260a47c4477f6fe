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

// Work plan of a W8A8 launch.  Query blocks of 256 rows are numbered
// head-major.  Blocks below split_from run whole, one workgroup of 32 rows a
// wave; every later one as two workgroups of 128 rows, 16 a wave (an end block
// of at most 128 rows leaves its second one empty).  Neither changes a row's
// arithmetic.  Causal workgroups are numbered by query block from the last,
// longest one to the first, heads fastest.
struct W8Plan {
    uint32_t nqb;         // query blocks of a head
    uint32_t bh;          // batch * hq
    uint32_t split_from;  // first block that runs as two workgroups (causal: all or none)
    uint32_t in_order;    // workgroups in the order of the blocks, whatever their XCD
};

struct W8Place {
    uint32_t bh, qb, half;  // batch * head, query block, its first or second 128 rows
    bool whole;             // all 256 rows
};

// kMode: 0 every block whole, 1 every block in two, 2 both.
template <bool kCausal, int kMode>
TU_HOST_DEVICE W8Place w8_place(const W8Plan &plan, uint32_t id) {
    W8Place p{0, 0, 0, kMode == 0};
    if (kCausal && !plan.in_order) {
        p.bh = id % plan.bh;
        id /= plan.bh;
        if constexpr (kMode == 1) {
            p.half = 1 - (id & 1);  // the later rows are the longer ones
            id >>= 1;
        }
        p.qb = plan.nqb - 1 - id;
        return p;
    }
    const uint32_t blocks = plan.nqb * plan.bh;
    if constexpr (kMode == 2) p.whole = id < plan.split_from;
    if (p.whole) {
        if (!plan.in_order) id = xcd_chunk(id, kMode == 0 ? blocks : plan.split_from);
    } else {
        const uint32_t from = kMode == 1 ? 0 : plan.split_from;
        id -= from;
        if (!plan.in_order) id = xcd_chunk(id, 2 * (blocks - from));
        p.half = id & 1;
        id = from + (id >> 1);
    }
    p.bh = id / plan.nqb;
    p.qb = id % plan.nqb;
    return p;
}

constexpr int64_t kW8BlockRows = 256, kW8TileKeys = 64;

// Time of causal workgroups of `rows` rows over all query blocks on `cus`
// compute units, in key tiles of one: the longest start first, so the time is
// their even share, or that of the rounds that hold all blocks of some length
// and longer.  `fixed` is a workgroup's time beside its tiles.
inline double w8_causal_time(const W8Plan &p, int64_t lq, int64_t lk, int64_t rows, double fixed, int64_t cus) {
    double even = 0.0, rounds = 0.0;
    int64_t count = 0;
    for (int64_t i = (lq + rows - 1) / rows; i > 0; --i) {
        const int64_t keys = std::min(lk, i * rows);
        const double t = static_cast<double>((keys + kW8TileKeys - 1) / kW8TileKeys) + fixed;
        count += p.bh;
        even += t * p.bh;
        rounds = std::max(rounds, static_cast<double>((count + cus - 1) / cus) * t);
    }
    return std::max(even / static_cast<double>(cus), rounds);
}

// Workgroups of 128 rows read K and V^T once for half the rows: a tile takes
// 1.22 us against 2.0 of a whole block's, and 6.3 us are spent beside the
// tiles against 9.  They pay where whole blocks leave compute units idle:
//   non-causal, the blocks past the last full round when they are at most
//     half a round: B1 H12 L1560 (84 blocks) 61.5 -> 37 us, H56 L4096 (896)
//     509 -> 461, B1 H12 L8190 (384) 461 -> 368; with more left over, two
//     half rounds are slower than one whole one (H60 L4096, 192 left: 512 and
//     531 us).  After full rounds the kernel for both forms takes more
//     than halves of a single key tile save;
//   causal, every block when the time by w8_causal_time is less: H4 L4001 117
//     -> 72 us, H40 L1000 41 -> 26, H12 L1560 x 512 25 -> 16; B2 H16 L4001
//     stays whole (149 against 166), and so does H10 L5000 x 128 (14.8 against
//     16.3: all blocks have two tiles, one round of whole ones against two).
// In a single round of blocks a head's workgroups run on all XCDs where they
// have at most four key tiles, or are at least 16: on one XCD they read the
// same key tile at once, and there is little to share from its L2 (B1 H3
// L20000 x 256 18.4 us on all XCDs, 19.0 on one, x 1024 42.9 and 43.2).  Over
// several rounds those of more than one tile stay on one (B1 H40 L7800 x 256
// 81.9 us, 83.7 on all; B1 H9 L8190 x 16 22.3, 22.0).
// Causal blocks of at most four tiles are equally long and go in order, as do
// whole ones of a single round, which all start at once (B2 H8 L4096 x 320
// 21.7 us from the longest on, 21.0 in order).
inline W8Plan w8_plan(int64_t batch, int64_t hq, int64_t lq, int64_t lk, bool causal, int64_t cus) {
    W8Plan p{static_cast<uint32_t>((lq + kW8BlockRows - 1) / kW8BlockRows), static_cast<uint32_t>(batch * hq), 0xffffffffu, 0};
    const int64_t blocks = static_cast<int64_t>(p.nqb) * p.bh;
    const bool few_keys = lk <= 4 * kW8TileKeys;
    p.in_order = causal ? few_keys : blocks <= cus ? few_keys || p.nqb >= 16 : lk <= kW8TileKeys;
    if (!causal) {
        const int64_t full = blocks / cus * cus;
        if (full < 0x7fffffff && 2 * (blocks - full) <= cus && (full == 0 || lk > kW8TileKeys))
            p.split_from = static_cast<uint32_t>(full);
        return p;
    }
    if (blocks >= 8 * cus) return p;  // an even share longer than any block
    if (0.58 * w8_causal_time(p, lq, lk, kW8BlockRows / 2, 5.2, cus) < w8_causal_time(p, lq, lk, kW8BlockRows, 4.5, cus))
        p.split_from = 0;
    else if (blocks <= cus)
        p.in_order = 1;
    return p;
}

// Workgroups of a launch.
inline int64_t w8_grid(const W8Plan &plan) {
    const int64_t blocks = static_cast<int64_t>(plan.nqb) * plan.bh;
    const int64_t whole = std::min<int64_t>(plan.split_from, blocks);
    return whole + 2 * (blocks - whole);
}

}  // namespace tu
