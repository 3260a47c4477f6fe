"""The SwiGLU quantizer by table (csrc/convrot_quant.hip): every bf16 gate
value, and passes that mix gates inside and outside the table, against the CPU
oracle bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests import inputs

pytestmark = pytest.mark.gpu


def _quantize(x, group):
    q, s = torch.ops.turing_utils.bf16_int8_convrot_quantize(x, group, swiglu=True)
    return q.cpu().numpy(), s.cpu().numpy().reshape(-1)


@pytest.mark.parametrize("group", [128, 256])
def test_every_gate(gpu_device, group):
    """All 65536 gate bit patterns: the finite ones a row per exponent (so that
    no row's scale hides the small ones), infinities and NaN last."""
    import comfyui_turing_utils_kernel.ops  # noqa: F401

    print(f"[silu table] every gate, group {group}", flush=True)
    k = 12544  # four waves, the last chunk ragged
    g = torch.Generator().manual_seed(3)
    rows = []
    for exponent in range(256):
        gates = torch.arange(128, dtype=torch.int32) + (exponent << 7)
        gates = torch.cat([gates, gates + 0x8000])
        row = gates[torch.randint(0, 256, (k,), generator=g)]
        row[:256] = gates
        rows.append(row)
    gate = torch.stack(rows).to(torch.int16).view(torch.bfloat16)
    up = torch.randn(256, k, generator=g).to(torch.bfloat16)
    x = torch.cat([gate, up], 1)
    q, s = _quantize(x.to(gpu_device), group)
    rq, rs = oracle.convrot_quant(inputs.bits(x), group, act=2)
    np.testing.assert_array_equal(s.view(np.uint32)[:255], rs.reshape(-1).view(np.uint32)[:255])
    np.testing.assert_array_equal(q[:255], rq[:255])
    # infinities and NaN: the codes alone (a NaN's payload is unspecified)
    np.testing.assert_array_equal(np.isnan(s[255:]), np.isnan(rs.reshape(-1)[255:]))


@pytest.mark.parametrize("rows,k,group", [(1, 12544, 256), (513, 8448, 256), (769, 14336, 256), (2050, 8320, 128), (515, 20480, 128),
                                          (300, 32768, 256)])
def test_rows_and_widths(gpu_device, rows, k, group):
    """Workgroups of one and several rows, the last one short; a few gates
    outside the table (0, 2^-19, 200, -130) in some passes."""
    import comfyui_turing_utils_kernel.ops  # noqa: F401

    print(f"[silu table] rows={rows} k={k} group={group}", flush=True)
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, 2 * k, generator=g)
    for i, value in enumerate((0.0, 2.0 ** -19, 200.0, -130.0)):
        x[i % rows, (i * 1031) % k] = value
    x = x.to(torch.bfloat16)
    q, s = _quantize(x.to(gpu_device), group)
    some = sorted({0, 1 % rows, 2 % rows, 3 % rows, rows // 2, rows - 2 if rows > 1 else 0, rows - 1})
    rq, rs = oracle.convrot_quant(inputs.bits(x[some].contiguous()), group, act=2)
    np.testing.assert_array_equal(s[some].view(np.uint32), rs.reshape(-1).view(np.uint32))
    np.testing.assert_array_equal(q[some], rq)
