"""Host checks of the Sage attention's automatic work plan (csrc/sage_attn.hip):
the schedule of causal key ranges, the workgroup numbering, and the workspace."""
from __future__ import annotations

import os

import pytest

from comfyui_turing_utils_kernel import _lib
from tests.test_attn_numbering import places  # noqa: F401
from tests.test_attn_schedule import KBKEY, KBQ, check_schedule, kernel_program


@pytest.mark.parametrize("kernel", ["sage", "sage64"])
@pytest.mark.parametrize("lq,lk,seg", [(1100, 1100, 8), (2049, 2049, 8), (3000, 3000, 12), (2500, 1000, 8),
                                       (700, 3000, 8), (1025, 1025, 16)])
def test_causal_ranges(lq, lk, seg, kernel):
    """A causal block's ranges start at multiples of 4 tiles (one query block's
    keys).  One that ends before the diagonal is a non-causal range; the last
    is the unsplit causal block shifted by its first tile."""
    assert seg % 4 == 0
    for qb in range((lq + KBQ - 1) // KBQ):
        tiles = (min(lk, (qb + 1) * KBQ) + KBKEY - 1) // KBKEY
        for z in range((tiles + seg - 1) // seg):
            base = z * seg
            assert base <= qb * KBQ // KBKEY  # every row of the block sees the range's first key
            if base + seg < tiles:
                _, info = kernel_program(0, lq, lk, False, qb, kernel, z, seg)
                assert info == {"tiles": seg, "my_tiles": seg}
                assert (base + seg) * KBKEY <= min(lk, qb * KBQ)  # no key of it is masked for any row
                check_schedule(lq, lk, False, qb, kernel, z, seg)
            else:
                check_schedule(lq - base * KBKEY, lk - base * KBKEY, True, qb - base * KBKEY // KBQ, kernel)


@pytest.mark.parametrize("nqb,bh,full,parts", [(4, 3, 0, 2), (5, 7, 11, 3), (32, 12, 256, 2)])
def test_noncausal_numbering(places, nqb, bh, full, parts):  # noqa: F811
    """Workgroup number -> (block, range), by the kernel's own function: every
    whole block once, every range of every later block once."""
    want = [(b // nqb, b % nqb, 0, 1) for b in range(full)]
    want += [(b // nqb, b % nqb, z, 0) for z in range(parts) for b in range(full, nqb * bh)]
    assert sorted(places("sage", 0, nqb, bh, full, parts)) == sorted(want)


def test_workspace_plan():
    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail(f"{_lib.LIB_PATH} is missing: {_lib.BUILD_HINT}")
    lib = _lib.load()
    need = lambda b, h, lq, lk, d=128, causal=0, cus=256: lib.tu_sage_attn_workspace(b, h, lq, lk, d, causal, cus)  # noqa: E731
    # 384 blocks: one whole round, the other 128 in two ranges; their rows
    # start in the middle of nothing: block 256 is head 8's first
    assert need(1, 12, 8190, 8190) == 2 * 4 * 8190 * (128 + 2) * 4
    assert need(1, 40, 32760, 32760) == 0        # 20 full rounds
    assert need(1, 40, 8190, 8190) == 0          # 5 full rounds
    assert need(1, 12, 7800, 512) == 0           # 8 key tiles are not worth splitting
    assert need(2, 16, 4001, 4001, causal=1) == 0  # enough blocks: longest first is even
    assert need(1, 4, 4001, 4001, causal=1) > 0
    assert need(0, 1, 1, 1) == 0 and need(1, 1, 256, 4096, cus=0) == 0
    for b, h, lq, lk in ((1, 1, 256, 4096), (1, 3, 300, 50000), (1, 12, 8190, 8190), (2, 8, 1000, 2000)):
        for causal in (0, 1):
            # never more than 16 ranges of every row
            assert need(b, h, lq, lk, causal=causal) <= 16 * b * h * lq * (128 + 2) * 4


@pytest.mark.parametrize("batch,hq,hkv", [(65536, 1, 1), (1, 65536, 1), (1, 65536, 65536)])
def test_prologue_refuses_what_its_parts_refuse(batch, hq, hkv):
    """tu_sage_quant and tu_sage_v_prep take at most 65535 heads and batch
    entries; the shared prologue as well, before it looks for a device."""
    buf = 1 << 12  # aligned, never dereferenced: the refusal comes first
    need = _lib.load().tu_sage_prep_workspace(batch, hkv, 64, 64, 0)
    with pytest.raises(RuntimeError, match="grid too large"):
        _lib.call("tu_sage_prep", buf, buf, buf, batch, hq, hkv, 64, 64, 64, *(64,) * 9, 0, 128, 128, buf, 64, 64, 64,
                  buf, 64, 64, 64, buf, buf, buf, 64, None, need, None)
