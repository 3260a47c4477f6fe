"""The bf16 GELU quantizer's choice of a table and of the rows that share it
(csrc/convrot_quant.hip): one row to several per workgroup, the last workgroup
short, with and without the table, against the CPU oracle bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle
from tests import inputs

pytestmark = pytest.mark.gpu


def _quantize(x, group):
    import comfyui_turing_utils_kernel.ops  # noqa: F401

    q, s = torch.ops.turing_utils.gelu_int8_convrot_quantize(x, group)
    return q.cpu().numpy(), s.cpu().numpy().reshape(-1)


# on 256 CUs: no table, 1, 3, 4, 5, 6, 7 and 8 rows a workgroup, rows of one to eight waves
@pytest.mark.parametrize("rows,k,group", [(1, 128, 128), (515, 4096, 256), (1, 8960, 128), (513, 13824, 128),
                                          (2050, 13824, 256), (4097, 8960, 128), (6144, 4352, 128), (6145, 4352, 128),
                                          (8192, 1152, 128), (8193, 1152, 128), (3, 32768, 256), (257, 26880, 128),
                                          (4001, 16640, 128), (5001, 5120, 128), (6145, 8192, 256), (1561, 20480, 256)])
def test_rows_and_widths(gpu_device, rows, k, group):
    print(f"[gelu rows] rows={rows} k={k} group={group}", flush=True)
    x = torch.randn(rows, k, generator=torch.Generator().manual_seed(rows + k))
    x[rows // 2, k // 3] = 40.0
    x = x.to(torch.bfloat16)
    q, s = _quantize(x.to(gpu_device), group)
    some = sorted({r % rows for r in (0, 1, 2, 3, rows // 2, rows - 3, rows - 2, rows - 1)})
    rq, rs = oracle.convrot_quant(inputs.bits(x[some].contiguous()), group, staged=True, act=1)
    np.testing.assert_array_equal(s[some].view(np.uint32), rs.reshape(-1).view(np.uint32))
    np.testing.assert_array_equal(q[some], rq)


@pytest.mark.parametrize("k", [4096, 8960])  # without the table and with it
def test_every_finite_input(gpu_device, k):
    """A row per exponent, so that no row's scale hides the small values."""
    print(f"[gelu rows] every input, k={k}", flush=True)
    g = torch.Generator().manual_seed(4)
    rows = []
    for exponent in range(255):
        values = torch.arange(128, dtype=torch.int32) + (exponent << 7)
        values = torch.cat([values, values + 0x8000])
        row = values[torch.randint(0, 256, (k,), generator=g)]
        row[:256] = values
        rows.append(row)
    x = torch.stack(rows).to(torch.int16).view(torch.bfloat16)
    q, s = _quantize(x.to(gpu_device), 128)
    rq, rs = oracle.convrot_quant(inputs.bits(x), 128, staged=True, act=1)
    np.testing.assert_array_equal(s.view(np.uint32), rs.reshape(-1).view(np.uint32))
    np.testing.assert_array_equal(q, rq)
