"""The Sage prologue in one call (tu_sage_prep) against its parts (K mean, Q / K
quantizers, V transpose): the same bits at block, chunk and tile edges, with
the mean added in the K blocks (up to 64 chunks) and by its own launch."""
from __future__ import annotations

import pytest
import torch

from comfyui_turing_utils_kernel.turing_sage import quant
from tests import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,hkv,lq,lk,d,blkq,blkk,smooth,layout", [
    (1, 1, 1, 1, 1, 64, 128, 128, True, "HND"),
    (2, 8, 2, 257, 300, 64, 128, 128, True, "NHD"),
    (1, 3, 3, 127, 129, 128, 16, 64, True, "HND"),
    (2, 2, 1, 64, 65, 128, 32, 64, False, "NHD"),
    (1, 2, 2, 1000, 8192, 128, 64, 128, True, "HND"),   # 64 chunks: the last that K blocks add themselves
    (1, 2, 2, 200, 8193, 64, 128, 64, True, "NHD"),     # 65: a launch of its own
    (3, 2, 2, 130, 20000, 128, 128, 128, True, "HND"),
])
def test_prologue_equals_its_parts(gpu_device, b, h, hkv, lq, lk, d, blkq, blkk, smooth, layout):
    print(f"[sage prep] b={b} h={h}/{hkv} lq={lq} lk={lk} d={d} blk=({blkq},{blkk}) {smooth} {layout}", flush=True)
    q, _, _ = inputs.attention(b, h, lq, d, lq)
    _, k, v = inputs.attention(b, hkv, lk, d, lk)
    to = (lambda t: t.transpose(1, 2).contiguous()) if layout == "NHD" else (lambda t: t)
    q, k, v = (to(t).to(gpu_device) for t in (q, k, v))
    got = quant.sage_prologue(q, k, v, blkq, blkk, layout, smooth)
    want = (*quant.per_block_int8(q, k, blkq, blkk, layout, smooth)[:4], quant.value_transpose(v, layout)[0])
    for name, x, y in zip(("q_int8", "q_scale", "k_int8", "k_scale", "value_t"), got, want):
        assert x.dtype == y.dtype and torch.equal(x, y), name


def test_prologue_takes_strided_views(gpu_device):
    """q, k and v as slices of one projection's output, as a Wan block has them."""
    qkv = torch.randn(1, 333, 3, 4, 128, generator=torch.Generator().manual_seed(5)).to(gpu_device, torch.bfloat16)
    q, k, v = qkv.unbind(2)
    got = quant.sage_prologue(q, k, v, tensor_layout="NHD")
    want = quant.sage_prologue(q.contiguous(), k.contiguous(), v.contiguous(), tensor_layout="NHD")
    assert all(torch.equal(x, y) for x, y in zip(got, want))
