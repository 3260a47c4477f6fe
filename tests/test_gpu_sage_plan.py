"""The automatic work plan of the Sage attention (tu_sage_attn_fwd_auto):
grids with a split last round, causal grids with split long rows, and the
causal block order, against the oracle and the unsplit kernel."""
from __future__ import annotations

import pytest
import torch

from comfyui_turing_utils_kernel import _lib
from comfyui_turing_utils_kernel.turing_sage import core
from comfyui_turing_utils_kernel.turing_sage.correctness import attention_error_metrics, require_attention_correctness
from tests import inputs
from tests.test_gpu_sage import GATE, _oracle_rows, _sample_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,hkv,lq,lk,d,causal", [
    (1, 2, 2, 257, 1025, 128, False),     # 4 blocks, all split, ragged rows and keys
    (1, 1, 1, 100, 4096, 64, False),      # one block in many ranges
    (2, 40, 40, 1000, 1030, 128, False),  # 320 blocks: one whole round, 64 split from mid-head
    (1, 300, 100, 256, 1500, 64, False),  # GQA, 300 one-block heads, 44 split
    (1, 2, 1, 3000, 3000, 128, True),     # causal: long rows split, the first blocks whole
    (2, 4, 2, 2049, 2049, 64, True),      # a last query block of one row
    (1, 3, 3, 2500, 1000, 128, True),     # more queries than keys
    (1, 3, 3, 700, 3000, 128, True),      # more keys than queries
    (2, 160, 160, 600, 600, 128, True),   # many heads: whole blocks, longest first
])
def test_auto_plan(gpu_device, b, h, hkv, lq, lk, d, causal):
    print(f"[attn plan] b={b} h={h} hkv={hkv} lq={lq} lk={lk} d={d} causal={causal}", flush=True)
    q, _, _ = inputs.attention(b, h, lq, d, 700 + lq)
    _, k, v = inputs.attention(b, hkv, lk, d, 800 + lk)
    state = core.prequantize_sageattn(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), "HND", is_causal=causal)
    args = (state.query_int8, state.query_scale, state.key_int8, state.key_scale, state.value_t)
    kw = dict(tensor_layout="HND", sm_scale=d ** -0.5, is_causal=causal)
    out = core.attention_from_vt(*args, **kw)
    whole = core.attention_from_vt(*args, **kw, kv_splits=1)
    nbytes = _lib.load().tu_sage_attn_workspace(b, h, lq, lk, d, int(causal), core._compute_units(gpu_device))
    torch.cuda.synchronize(gpu_device)
    rows = _sample_rows(b, h, lq, 96, lq + lk)
    ref = torch.from_numpy(_oracle_rows(q, k, v, rows, 128, 128, causal, d ** -0.5))
    got = out.float().cpu()[rows[:, 0], rows[:, 1], rows[:, 2]]
    require_attention_correctness(attention_error_metrics(got, ref, candidate_name="plan", reference_name="oracle"),
                                  **GATE)
    # against the unsplit kernel: the fp32 merge, and P rounded to bf16
    # against each range's own base
    both = attention_error_metrics(out.float().cpu().flatten(1), whole.float().cpu().flatten(1),
                                   candidate_name="plan", reference_name="whole")
    assert both.cosine >= 0.99999 and both.max_abs <= 1e-2
    if nbytes == 0:
        assert torch.equal(out, whole)
        return
    # stale workspace contents change nothing
    ws = torch.full((nbytes // 4,), float("nan"), dtype=torch.float32, device=gpu_device)
    again = torch.empty_like(whole)
    lengths = [t.stride(i) for t in (state.query_int8, state.key_int8, again) for i in (0, 1, 2)]
    call = lambda o, w, n: _lib.call(  # noqa: E731
        "tu_sage_attn_fwd_auto", state.query_int8.data_ptr(), state.query_scale.data_ptr(), 128,
        state.key_int8.data_ptr(), state.key_scale.data_ptr(), 128, state.value_t.data_ptr(),
        state.value_t.shape[-1], o.data_ptr(), b, h, hkv, lq, lk, d, *lengths, d ** -0.5, int(causal),
        core._compute_units(gpu_device), w, n, _lib.stream_of(gpu_device))
    call(again, ws.data_ptr(), nbytes)
    assert torch.equal(again, out)
    # a workspace too small for any split runs whole
    call(again, ws.data_ptr(), 16)
    assert torch.equal(again, whole)


@pytest.mark.parametrize("d", [64, 128])
def test_output_rows_on_8_byte_boundaries(gpu_device, d):
    """The C ABI takes output rows aligned to 8 bytes: the same bits as with
    16-byte rows, and nothing written between the rows."""
    q, k, v = inputs.attention(1, 2, 300, d, 31)
    state = core.prequantize_sageattn(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device))
    args = (state.query_int8, state.query_scale, state.key_int8, state.key_scale, state.value_t)
    want = core.attention_from_vt(*args)
    wide = torch.full((1, 2, 300, d + 4), 7.0, dtype=torch.bfloat16, device=gpu_device)
    core.attention_from_vt(*args, output=wide[..., :d])
    assert torch.equal(wide[..., :d], want) and bool((wide[..., d:] == 7.0).all())


def test_misaligned_workspace(gpu_device):
    """A workspace that a split call needs is refused off 16 bytes; where none
    is needed it is not used."""
    for lk, needed in ((4096, True), (300, False)):
        q, k, v = inputs.attention(1, 2, lk, 128, 7)
        state = core.prequantize_sageattn(q[:, :, :200].contiguous().to(gpu_device), k.to(gpu_device), v.to(gpu_device))
        args = (state.query_int8, state.query_scale, state.key_int8, state.key_scale, state.value_t)
        cus = core._compute_units(gpu_device)
        splits = _lib.load().tu_sage_attn_kv_splits(1, 2, 200, lk, 0, cus)
        assert (splits > 1) == needed
        ws = torch.zeros(core.split_workspace_bytes(1, 2, 200, lk, 128, splits) // 4 + 1, dtype=torch.float32, device=gpu_device)[1:]
        if needed:
            with pytest.raises(RuntimeError, match="aligned"):
                core.attention_from_vt(*args, workspace=ws)
        else:
            assert torch.equal(core.attention_from_vt(*args, workspace=ws), core.attention_from_vt(*args))
            assert not ws.any()
