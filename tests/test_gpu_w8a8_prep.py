"""The fused W8A8 prologue (tu_w8a8_prep) gives the codes, scales and anchors'
effect of the separate quantizers, bit for bit, head_dim 64 padded to 128."""
from __future__ import annotations

import pytest
import torch

from tests.test_gpu_w8a8 import _qkv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("b,hq,hk,lq,lk,rotate,stabilize", [
    (1, 1, 1, 1, 1, True, True),
    (2, 4, 2, 63, 65, True, False),
    (1, 3, 3, 129, 2049, False, False),    # 17 chunks of 121 tokens, the last one short
    (1, 70, 70, 65, 2300, True, True),     # enough heads for the fewest chunks
    (1, 1, 1, 40, 9000, True, True),       # the most chunks
])
def test_matches_separate_quantizers(gpu_device, dtype, d, b, hq, hk, lq, lk, rotate, stabilize):
    from comfyui_turing_utils_kernel.turing_sage.quant import per_warp_int8_hadamard, quantize_v_int8, w8a8_prologue

    print(f"[w8a8-prep] {dtype} d={d} b={b} hq={hq} hk={hk} lq={lq} lk={lk}", flush=True)
    q, k, v = (t.to(gpu_device) for t in _qkv(b, hq, hk, lq, lk, d, dtype, lq + lk + d))
    # V as an HND view of NHD rows
    v = v.transpose(1, 2).contiguous().transpose(1, 2)
    want = [*per_warp_int8_hadamard(q, k, stabilize_k=stabilize, rotate=rotate), *quantize_v_int8(v)]
    got = w8a8_prologue(q, k, v, stabilize_k=stabilize, rotate=rotate)
    pad = 128 - d
    for i, channels in ((0, (0, pad)), (2, (0, pad)), (4, (0, 0, 0, pad))):
        want[i] = torch.nn.functional.pad(want[i], channels)
    want[5] = torch.nn.functional.pad(want[5], (0, pad), value=1.0e-12)
    for name, x, y in zip(("q", "q_scale", "k", "k_scale", "v", "v_scale"), got, want):
        assert x.shape == y.shape and torch.equal(x, y), name
