"""Workgroup numbers of the attention kernels -> their query blocks, by the
functions that the kernels themselves call (csrc/attn_plan.h), compiled for the
host: every part of every block once, whatever the grid's remainder by 8."""
from __future__ import annotations

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "comfyui-turing-utils_amd", "csrc")
PROGRAM = r"""
#include "attn_plan.h"
#include <cstdio>
#include <cstdlib>
#include <cstring>
using namespace tu;
template <bool kCausal, bool kSplit> void sage(const AttnPlan &p) {
    for (uint32_t i = 0; i < sage_grid<kCausal>(p); ++i) {
        const SagePlace w = sage_place<kCausal, kSplit>(p, i);
        std::printf("%u %u %u %d\n", w.bh, w.qb, w.z, int(w.whole));
    }
}
template <bool kCausal, int kMode> void w8(const W8Plan &p) {
    for (uint32_t i = 0; i < w8_grid(p); ++i) {
        const W8Place w = w8_place<kCausal, kMode>(p, i);
        std::printf("%u %u %u %d\n", w.bh, w.qb, w.half, int(w.whole));
    }
}
int main(int, char **v) {
    if (!std::strcmp(v[1], "w8plan")) {
        const W8Plan p = w8_plan(std::atoi(v[2]), std::atoi(v[3]), std::atoi(v[4]), std::atoi(v[5]), v[6][0] == '1', 256);
        std::printf("%u %u %u %u\n", p.nqb, p.bh, p.split_from, p.in_order);
        return 0;
    }
    const uint32_t nqb = std::atoi(v[3]), bh = std::atoi(v[4]), from = std::atoi(v[5]), parts = std::atoi(v[6]);
    const bool causal = v[2][0] == '1';
    if (!std::strcmp(v[1], "sage")) {
        AttnPlan p{};
        p.nqb = nqb, p.bh = bh, p.split_from = from, p.parts = parts;
        if (causal) parts > 1 ? sage<true, true>(p) : sage<true, false>(p);
        else parts > 1 ? sage<false, true>(p) : sage<false, false>(p);
    } else {
        W8Plan p{};
        p.nqb = nqb, p.bh = bh, p.split_from = from, p.in_order = parts;
        if (causal) from ? w8<true, 0>(p) : w8<true, 1>(p);
        else if (from >= nqb * bh) w8<false, 0>(p);
        else from ? w8<false, 2>(p) : w8<false, 1>(p);
    }
}
"""


@pytest.fixture(scope="module")
def places(tmp_path_factory):
    d = tmp_path_factory.mktemp("numbering")
    (d / "numbering.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-O1", "-I", CSRC, str(d / "numbering.cpp"), "-o", str(d / "numbering")],
                   check=True, timeout=120)

    def run(*args):
        out = subprocess.run([str(d / "numbering"), *map(str, args)], check=True, capture_output=True, text=True, timeout=60)
        return [tuple(map(int, ln.split())) for ln in out.stdout.splitlines()]

    return run


GRIDS = [(4, 3), (5, 7), (1, 1), (1, 40), (33, 1), (31, 12), (17, 16)]


@pytest.mark.parametrize("nqb,bh", GRIDS)
def test_sage_noncausal(places, nqb, bh):
    blocks = [(b, q) for b in range(bh) for q in range(nqb)]
    n = len(blocks)
    assert sorted(places("sage", 0, nqb, bh, 0xFFFFFF, 1)) == [(b, q, 0, 1) for b, q in blocks]
    for full in sorted({0, n // 2, n - 1}):
        for parts in (2, 3, 7, 16):
            got = places("sage", 0, nqb, bh, full, parts)
            assert sorted(got[:full]) == [(b, q, 0, 1) for b, q in blocks[:full]]
            # all first ranges before any second, blocks in turn over the XCDs
            assert got[full:] == [(b, q, z, 0) for z in range(parts) for b, q in blocks[full:]]


@pytest.mark.parametrize("nqb,bh", GRIDS)
def test_sage_causal(places, nqb, bh):
    for parts in (1, 2, 5, 16):
        got = places("sage", 1, nqb, bh, 0, parts)
        assert sorted(w[:3] for w in got) == sorted((b, q, z) for b in range(bh) for q in range(nqb) for z in range(parts))
        assert [w[1] for w in got] == sorted((w[1] for w in got), reverse=True)  # the longest blocks start first


@pytest.mark.parametrize("nqb,bh", GRIDS)
def test_w8a8_noncausal(places, nqb, bh):
    blocks = [(b, q) for b in range(bh) for q in range(nqb)]
    n = len(blocks)
    for full in sorted({0, n // 2, n - 1, n}):
        want = [(b, q, 0, 1) for b, q in blocks[:full]], [(b, q, h, 0) for b, q in blocks[full:] for h in (0, 1)]
        got = places("w8", 0, nqb, bh, full, 0)
        assert (sorted(got[:full]), sorted(got[full:])) == want
        got = places("w8", 0, nqb, bh, full, 1)  # in order
        assert (got[:full], got[full:]) == want


@pytest.mark.parametrize("nqb,bh", GRIDS)
def test_w8a8_causal(places, nqb, bh):
    blocks = [(b, q) for b in range(bh) for q in range(nqb)]
    assert sorted(places("w8", 1, nqb, bh, 0xFFFFFF, 0)) == [(b, q, 0, 1) for b, q in blocks]
    assert places("w8", 1, nqb, bh, 0xFFFFFF, 1) == [(b, q, 0, 1) for b, q in blocks]
    assert places("w8", 1, nqb, bh, 0, 1) == [(b, q, h, 0) for b, q in blocks for h in (0, 1)]
    got = places("w8", 1, nqb, bh, 0, 0)
    assert sorted(got) == sorted((b, q, h, 0) for b in range(bh) for q in range(nqb) for h in (0, 1))
    rows = [2 * q + h for _, q, h, _ in got]
    assert rows == sorted(rows, reverse=True)  # the longest first


WHOLE = 0xFFFFFFFF


@pytest.mark.parametrize("b,h,lq,lk,causal,split_from,in_order", [
    (1, 12, 1560, 512, 0, 0, 0),            # 84 blocks: halves 16 us, whole 25
    (1, 12, 8190, 8190, 0, 256, 0),         # 384: 368 us, whole 461
    (1, 60, 4096, 4096, 0, WHOLE, 0),       # 192 left over: whole 512, halves 531
    (1, 12, 7800, 64, 0, WHOLE, 1),         # one key tile: the kernel of both forms is slower
    (1, 12, 7800, 65, 0, 256, 0),
    (1, 3, 20000, 256, 0, WHOLE, 1),        # 18.4 us in order, 19.0 by XCD
    (1, 3, 20000, 1024, 0, WHOLE, 1),
    (1, 40, 7800, 256, 0, WHOLE, 0),        # several rounds: 81.9 by XCD, 83.7 in order
    (1, 4, 4001, 4001, 1, 0, 0),            # 72 us, whole 117
    (1, 40, 1000, 1000, 1, 0, 0),           # 26, whole 41
    (1, 12, 1560, 512, 1, 0, 0),            # 16, whole 25
    (2, 16, 4001, 4001, 1, WHOLE, 0),       # 149, halves 166
    (2, 5, 5000, 128, 1, WHOLE, 1),         # two tiles each: 14.6, halves 16.3
    (2, 24, 1024, 512, 1, WHOLE, 1),        # 26.6, halves 27.8
    (2, 24, 1024, 1024, 1, 0, 0),           # 28.4, whole 41.5
    (1, 12, 5000, 1024, 1, WHOLE, 1),       # 43.2, halves 48.1
    (1, 40, 1560, 256, 1, 0, 1),            # 25.1, whole 29.6
])
def test_w8a8_plan(places, b, h, lq, lk, causal, split_from, in_order):
    """On 256 CUs, at sizes where both sides were measured."""
    assert places("w8plan", b, h, lq, lk, causal) == [(-(-lq // 256), b * h, split_from, in_order)]
