"""The native host calls (csrc/host_calls.cpp) give the general route's bits,
and step aside (return None) for every call that is not plain."""
from __future__ import annotations

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from comfyui_turing_utils_kernel import _lib, integration
from comfyui_turing_utils_kernel.turing_sage import core
from tests import inputs

pytestmark = pytest.mark.gpu

REAL = _lib.host_calls


class _General:
    """Every native call refused: the general route alone."""

    def __getattr__(self, name):
        return lambda *args: None


@pytest.fixture
def both(monkeypatch):
    def run(f):
        served = []

        class Spy:
            def __getattr__(self, name):
                def call(*args):
                    served.append(getattr(REAL(), name)(*args))
                    return served[-1]
                return call

        monkeypatch.setattr(_lib, "host_calls", Spy)
        native = f()
        monkeypatch.setattr(_lib, "host_calls", _General)
        general = f()
        monkeypatch.setattr(_lib, "host_calls", REAL)
        return native, general, [s is not None for s in served]
    return run


def _linear(dev, rows=(3, 7), k=512, n=136, act=None):
    width = 2 * k if act == "swiglu" else k
    m = rows if isinstance(rows, int) else rows[0] * rows[1]
    x = inputs.activation(m, width, 1).to(dev).reshape(*((rows,) if isinstance(rows, int) else rows), width)
    w, ws, bias = (t.to(dev) for t in inputs.weights(n, k, 1))
    return x, w, ws.float().reshape(-1), bias.float()


@pytest.mark.parametrize("act", [None, "none", "gelu_tanh", "swiglu"])
@pytest.mark.parametrize("out_dtype", [None, torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("group,with_bias", [(128, True), (256, False)])
def test_linear(gpu_device, both, act, out_dtype, group, with_bias):
    x, w, ws, bias = _linear(gpu_device, act=act)
    native, general, served = both(lambda: integration.int8_linear(
        x, w, ws, bias if with_bias else None, out_dtype, True, group, act))
    assert served == [True] and native.dtype == general.dtype and native.shape == general.shape == (3, 7, 136)
    assert torch.equal(native, general)


@pytest.mark.parametrize("act", [None, "swiglu"])
def test_rows_too_wide_for_the_quantizer(gpu_device, act):
    """The general route's error, with the module and without."""
    x, w, ws, bias = _linear(gpu_device, rows=1, k=65536 + 256, n=8, act=act)
    with pytest.raises(ValueError, match="65536-column limit"):
        integration.int8_linear(x, w, ws, bias, None, True, 256, act)


def test_linear_forms_that_are_not_plain(gpu_device, both):
    x, w, ws, bias = _linear(gpu_device, rows=8)
    off = torch.empty(8 * 512 + 1, dtype=torch.bfloat16, device=gpu_device)[1:].reshape(8, 512).copy_(x)
    for name, args in {
        "misaligned": (off, w, ws, bias), "strided x": (x.repeat(1, 2)[:, :512], w, ws, bias),
        "strided w": (x, w.repeat(1, 2)[:, :512], ws, bias), "scalar scale": (x, w, ws[:1], bias),
        "bf16 bias": (x, w, ws, bias.bfloat16()), "host scale": (x, w, ws.cpu(), bias),
    }.items():
        native, general, served = both(lambda: integration.int8_linear(*args, None, True, 128))
        assert served == [False] and torch.equal(native, general), name
    plain = integration.int8_linear(x, w, ws, bias, None, True, 128)
    param = torch.nn.Parameter(w, requires_grad=False)
    native, _, served = both(lambda: integration.int8_linear(x, param, ws, bias, None, True, 128))
    assert served == [True] and torch.equal(native, plain)
    with torch.inference_mode():
        native, _, served = both(lambda: integration.int8_linear(x.clone(), w, ws, bias, None, True, 128))
    assert served == [True] and torch.equal(native, plain)
    leaf = x.clone().requires_grad_()
    native, general, served = both(lambda: integration.int8_linear(leaf, w, ws, bias, None, True, 128))
    assert served == [False] and native.requires_grad == general.requires_grad
    with torch.no_grad():
        native, _, served = both(lambda: integration.int8_linear(leaf, w, ws, bias, None, True, 128))
    assert served == [True] and torch.equal(native, plain)

    class Dispatch(TorchDispatchMode):
        seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Dispatch(), Function()):
        with mode:
            native, general, served = both(lambda: integration.int8_linear(x, w, ws, bias, None, True, 128))
        assert not any(served) and torch.equal(native, plain)
    assert any("int8_linear" in s for s in Dispatch.seen)
    with pytest.raises(ValueError, match="scalar or have 136 values"):
        integration.int8_linear(x, w, ws[:100], bias, None, True, 128)
    with pytest.raises(ValueError):
        integration.int8_linear(x, w[:, :256], ws, bias, None, True, 128)
    compiled = torch.compile(lambda a: integration.int8_linear(a, w, ws, bias, None, True, 128), backend="eager",
                             fullgraph=False)
    assert torch.equal(compiled(x), plain)


@pytest.mark.parametrize("layout", ["HND", "NHD"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal,smooth,blkq,blkk,scale", [(False, True, 128, 128, None), (True, False, 64, 64, 0.11)])
def test_sage(gpu_device, both, layout, d, causal, smooth, blkq, blkk, scale):
    q, _, _ = (t.to(gpu_device) for t in inputs.attention(2, 4, 300, d, 3))
    _, k, v = (t.to(gpu_device) for t in inputs.attention(2, 2, 1100, d, 4))
    if layout == "NHD":
        q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, v))
    native, general, served = both(lambda: core.sageattn(q, k, v, layout, causal, scale, smooth, blkq, blkk))
    assert served == [True] and torch.equal(native, general) and native.stride() == general.stride()
    # HND views of NHD rows and back
    other = "NHD" if layout == "HND" else "HND"
    native, general, served = both(lambda: core.sageattn(*(t.transpose(1, 2) for t in (q, k, v)), other, causal, scale,
                                                         smooth, blkq, blkk))
    assert served == [True] and torch.equal(native, general) and native.stride() == general.stride()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("causal,rotate,stabilize", [(False, True, True), (True, False, True), (False, True, False)])
def test_w8a8(gpu_device, both, dtype, d, causal, rotate, stabilize):
    q, _, _ = (t.to(gpu_device, dtype) for t in inputs.attention(2, 4, 130, d, 3))
    _, k, v = (t.to(gpu_device, dtype) for t in inputs.attention(2, 2, 333, d, 4))
    native, general, served = both(lambda: core.w8a8attn(q, k, v, is_causal=causal, rotate_qk=rotate,
                                                         stabilize_k=stabilize))
    assert served == [True] and torch.equal(native, general)
    assert native.stride() == general.stride() and native.dtype == dtype


def test_attention_forms_that_are_not_plain(gpu_device, both):
    q, k, v = (t.to(gpu_device) for t in inputs.attention(1, 2, 100, 128, 5))
    for f in (lambda: core.sageattn(q[..., :96], k[..., :96], v[..., :96]),
              lambda: core.sageattn(q.half(), k.half(), v.half()),
              lambda: core.w8a8attn(q[..., :80], k[..., :80], v[..., :80])):
        native, general, served = both(f)
        assert served == [False] and torch.equal(native, general)
    for call in (core.sageattn, core.w8a8attn):
        with pytest.raises(ValueError):
            call(q, k[:, :, :50], v)
        with pytest.raises(TypeError):
            call(q.float(), k.float(), v.float())
    with pytest.raises(ValueError, match="sm_scale"):
        core.sageattn(q, k, v, sm_scale=float("inf"))
    with pytest.raises(ValueError, match="key_tile_tokens"):
        core.w8a8attn(q, k, v, key_tile_tokens=96)


def test_on_a_side_stream_and_under_capture(gpu_device):
    x, w, ws, bias = _linear(gpu_device, rows=9)
    q, k, v = (t.to(gpu_device) for t in inputs.attention(1, 4, 700, 128, 6))
    calls = (lambda: integration.int8_linear(x, w, ws, bias, None, True, 128), lambda: core.sageattn(q, k, v),
             lambda: core.w8a8attn(q, k, v))
    want = [f() for f in calls]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = [f() for f in calls]
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = [f() for f in calls]
    for _ in range(3):
        for t in got:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_without_the_module(gpu_device, monkeypatch):
    """The three calls where the module does not load: the general route's results."""
    import sys

    import comfyui_turing_utils_kernel as package

    x, w, ws, bias = _linear(gpu_device, rows=9)
    q, k, v = (t.to(gpu_device) for t in inputs.attention(1, 4, 700, 128, 6))
    calls = (lambda: integration.int8_linear(x, w, ws, bias, None, True, 128), lambda: core.sageattn(q, k, v),
             lambda: core.w8a8attn(q, k, v))
    want = [f() for f in calls]
    monkeypatch.setattr(_lib, "_host", None)
    monkeypatch.delattr(package, "_host_calls", raising=False)
    monkeypatch.setitem(sys.modules, "comfyui_turing_utils_kernel._host_calls", None)
    with pytest.warns(RuntimeWarning, match="cannot be loaded"):
        got = [f() for f in calls]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
