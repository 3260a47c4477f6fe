"""The W8A8 attention's work plan (csrc/w8a8_attn.hip): whole blocks, half
blocks and grids with both give a row the same bits, whatever else is in the
launch, and match the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.test_gpu_w8a8 import _compare, _oracle_attention, _qkv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,lq,lk,dtype,causal", [
    (256, 130, 129, torch.bfloat16, False),   # one full round of whole blocks
    (300, 257, 200, torch.float16, False),    # 600 blocks: two rounds whole, 88 in two, every second one of one row
    (259, 256, 65, torch.bfloat16, False),    # three blocks past a round
    (200, 250, 130, torch.bfloat16, False),   # more than half a round left over: whole
    (256, 300, 300, torch.bfloat16, True),    # causal, whole blocks
    (16, 700, 300, torch.float16, True),      # causal, half blocks, more queries than keys
    (300, 257, 64, torch.bfloat16, False),    # one key tile over several rounds: whole, in order
    (12, 5000, 200, torch.float16, False),    # one round of many blocks of a head, in order
    (40, 700, 200, torch.bfloat16, True),     # causal, few keys: half blocks in order
    (240, 250, 200, torch.bfloat16, True),    # whole ones in order
    (16, 4096, 320, torch.float16, True),     # causal, one round of whole blocks, in order
])
def test_rows_do_not_depend_on_the_grid(gpu_device, h, lq, lk, dtype, causal):
    from comfyui_turing_utils_kernel.turing_sage import w8a8attn

    print(f"[w8a8-plan] h={h} lq={lq} lk={lk} {dtype} causal={causal}", flush=True)
    q, k, v = _qkv(1, h, h, lq, lk, 128, dtype, h + lq)
    qd, kd, vd = (t.to(gpu_device) for t in (q, k, v))
    out = w8a8attn(qd, kd, vd, is_causal=causal)
    heads = sorted({0, 1, h // 2, h - 45 if h > 45 else 2, h - 2, h - 1})
    few = w8a8attn(qd[:, heads], kd[:, heads], vd[:, heads], is_causal=causal)  # a grid of half blocks
    assert torch.equal(out[:, heads], few)
    rows = np.array([(0, i, r) for i in range(len(heads)) for r in sorted({0, 1, 127, 128, lq - 2, lq - 1})])
    ref = _oracle_attention(q[:, heads], k[:, heads], v[:, heads], causal, 128 ** -0.5, rows)
    _compare(few.cpu().float()[rows[:, 0], rows[:, 1], rows[:, 2]], ref)
