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


def _tile(device, m, n, k):
    """The tile of the launch, None on another number of CUs than the shapes were chosen for."""
    cus = torch.cuda.get_device_properties(device).multi_processor_count
    t = _lib.load().tu_int8_gemm_tile(m, n, k, cus)
    return (t >> 16, t & 0xFFFF) if cus == 256 else None


# K of 0 to 6 full 128-byte steps with and without a partial one, and long
@pytest.mark.parametrize("k", [16, 112, 128, 256, 272, 384, 512, 528, 640, 768, 5120])
# one tile of 64 x 64 and several (the first four), 128 x 64, 128 x 128, 128 x 192
@pytest.mark.parametrize("m,n", [(1, 8), (65, 72), (63, 1032), (130, 5128), (515, 2568), (515, 4104), (1000, 5000)])
def test_small_tiles_exact(gpu_device, m, n, k):
    tile = _tile(gpu_device, m, n, k)
    print(f"[gemm tiles] m={m} n={n} k={k} tile={tile}", flush=True)
    assert tile in (None, {2568: (128, 64), 4104: (128, 128), 5000: (128, 192)}.get(n, (64, 64)))
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


@pytest.mark.parametrize("m,n,k,want", [(1, 1032, 528, (64, 64)), (130, 5128, 640, (64, 64)), (515, 2568, 5120, (128, 64)),
                                        (515, 4104, 640, (128, 128)), (1000, 5000, 5120, (128, 192))])
def test_small_tile_epilogues(gpu_device, m, n, k, want):
    """Each output type and the gated residual against the 256 x 256 tile."""
    tile = _tile(gpu_device, m, n, k)
    print(f"[gemm tiles] epilogues m={m} n={n} k={k} tile={tile}", flush=True)
    assert tile in (None, want)
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
