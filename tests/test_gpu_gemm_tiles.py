"""The GEMM's small tiles (128 x 192, 128 x 128, 128 x 64, 64 x 64 with rings of
three and four K steps), which the automatic choice takes for grids that
larger tiles leave mostly idle: bit-exact against torch's integer product and
the 256 x 256 tile, on ragged rows and columns and around the ring's depth."""
from __future__ import annotations

import pytest
import torch

from comfyui_turing_utils_kernel import _lib
from tests import inputs

pytestmark = pytest.mark.gpu


def _rand_i8(shape, seed):
    return torch.randint(-128, 128, shape, generator=torch.Generator().manual_seed(seed), dtype=torch.int8)


# K of 0 to 6 full 128-byte steps with and without a partial one, and long
@pytest.mark.parametrize("k", [16, 112, 128, 256, 272, 384, 512, 528, 640, 768, 5120])
# one tile and less; 64 x 64; 128 x 64; 128 x 128; 128 x 192 (by K, on 256 CUs)
@pytest.mark.parametrize("m,n", [(1, 8), (65, 72), (63, 1032), (130, 5128), (515, 2568), (1000, 5000)])
def test_small_tiles_exact(gpu_device, m, n, k):
    print(f"[gemm tiles] m={m} n={n} k={k}", flush=True)
    a, w = _rand_i8((m, k), m + k), _rand_i8((n, k), n + k)
    ad, wd = a.to(gpu_device), w.to(gpu_device)
    got = torch.ops.turing_utils.int8_gemm_i32(ad, wd)
    ref = (a.double() @ w.double().T) if m * n * k < 2e9 else None  # exact: every sum is below 2^53
    if ref is not None:
        assert torch.equal(got.cpu().double(), ref)
    whole = torch.empty_like(got)  # the 256 x 256 tile
    _lib.call("tu_int8_gemm_ex", ad.data_ptr(), wd.data_ptr(), None, None, None, whole.data_ptr(), 3, m, n, k, 1,
              _lib.stream_of(gpu_device))
    assert torch.equal(got, whole)


@pytest.mark.parametrize("m,n,k", [(1, 1032, 528), (130, 5128, 640), (515, 2568, 5120), (1000, 5000, 5120)])
def test_small_tile_epilogues(gpu_device, m, n, k):
    """Each output type and the gated residual against the 256 x 256 tile."""
    print(f"[gemm tiles] epilogues m={m} n={n} k={k}", flush=True)
    dev = gpu_device
    a = _rand_i8((m, k), m).to(dev)
    w, ws, bias = (t.to(dev) for t in inputs.weights(n, k, 3))
    xs = torch.rand(m, generator=torch.Generator().manual_seed(1)).to(dev) * 1e-2
    for code, dtype in ((0, torch.bfloat16), (1, torch.float16), (2, torch.float32)):
        got = torch.ops.turing_utils.int8_linear_out(a, w, xs, ws, bias, dtype)
        whole = torch.empty_like(got)
        _lib.call("tu_int8_gemm_ex", a.data_ptr(), w.data_ptr(), xs.data_ptr(), ws.data_ptr(), bias.data_ptr(),
                  whole.data_ptr(), code, m, n, k, 1, _lib.stream_of(dev))
        assert torch.equal(got, whole), dtype
        if dtype == torch.bfloat16:
            y = got
    gen = torch.Generator().manual_seed(2)
    res, gate = (torch.randn(r, n, generator=gen).to(dev, torch.bfloat16) for r in (m, (m + 6) // 7))
    out = torch.ops.turing_utils.int8_linear_residual(a, w, xs, ws, bias, res, gate, 7)
    # the fp32 fma through fp64 (an exact product of two bf16), then bf16
    g = gate.double().repeat_interleave(7, 0)[:m]
    assert torch.equal(out, (y.double() * g + res.double()).float().to(torch.bfloat16))
