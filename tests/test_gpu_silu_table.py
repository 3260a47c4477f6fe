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


# on 256 CUs: 1, 3 and 4 rows a workgroup, and rows without a table (of three, five and eight waves, and four)
@pytest.mark.parametrize("rows,k,group", [(1, 12544, 256), (513, 8448, 256), (769, 14336, 256), (2050, 8320, 128), (515, 20480, 128),
                                          (300, 32768, 256), (515, 12416, 128), (2051, 16384, 256), (3001, 12544, 128)])
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


@pytest.mark.parametrize("rows,k,group", [(3, 14336, 256), (2050, 12544, 128)])
def test_gates_outside_the_table(gpu_device, rows, k, group):
    """Rows of zero gates of both signs (with finite, infinite and NaN up
    values), of gates around the table's ends, of single gates outside it, and
    ordinary rows, in turn."""
    import comfyui_turing_utils_kernel.ops  # noqa: F401

    print(f"[silu table] outside rows={rows} k={k} group={group}", flush=True)
    g = torch.Generator().manual_seed(rows + 1)
    gate = torch.randn(rows, k, generator=g)
    up = torch.randn(rows, k, generator=g)
    ends = torch.tensor([0.0, -0.0, 2.0 ** -133, -2.0 ** -126, 2.0 ** -25, -2.0 ** -24, 2.0 ** -24, 2.0 ** -23, 88.5, -88.5,
                         89.0, -89.0, 128.0, -130.0, 3e38, -3e38])
    for r in range(rows):
        kind = r % 6
        if kind == 0:
            gate[r] = torch.where(torch.arange(k) % 2 == 0, 0.0, -0.0)
        elif kind == 1:
            gate[r] = ends[torch.randint(0, 14, (k,), generator=g)]
        elif kind == 2:
            gate[r] = ends[torch.randint(0, 7, (k,), generator=g)]
        elif kind == 3:
            at = torch.arange(0, k, 1031)
            gate[r, at] = ends[torch.arange(at.numel()) % 16]
    x = torch.cat([gate, up], 1).to(torch.bfloat16)
    q, s = _quantize(x.to(gpu_device), group)
    some = [r for r in range(rows) if r < 12 or r >= rows - 8]
    rq, rs = oracle.convrot_quant(inputs.bits(x[some].contiguous()), group, act=2)
    np.testing.assert_array_equal(s[some].view(np.uint32), rs.reshape(-1).view(np.uint32))
    np.testing.assert_array_equal(q[some], rq)
    # a zero gate times an infinite or NaN up value is NaN, in this row alone
    x[0, k + 5] = float("inf")
    x[0, k + 2000] = float("nan")
    q2, s2 = _quantize(x.to(gpu_device), group)
    rq, rs = oracle.convrot_quant(inputs.bits(x[:1].contiguous()), group, act=2)
    np.testing.assert_array_equal(s2[:1].view(np.uint32), rs.reshape(-1).view(np.uint32))
    np.testing.assert_array_equal(q2[:1], rq)
    np.testing.assert_array_equal(q2[1:], q[1:])
