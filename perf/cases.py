"""The measured work of this package: what a quantized DiT runs through its public entry points.

Three kinds of call make up a model's time, and a fourth puts them together:

* ``linear``: ``integration.int8_linear``, the plugin's W8A8 linear (ConvRot quantizer, optionally with the
  input activation, then the INT8 GEMM), from one modulation row to a whole video's tokens;
* ``sage``: ``turing_sage.sageattn``, the Sage attention from bf16 Q / K / V, self- and cross-attention;
* ``w8a8``: ``turing_sage.w8a8attn``, the dense W8A8 attention;
* ``block``: ``wan_block.WanBlockW8A8``, one whole Wan 2.1 block forward.

The package is an inference path, so there is no backward direction.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "comfyui-turing-utils_amd"))

from comfyui_turing_utils_kernel import integration, turing_sage, wan_block  # noqa: E402

DEVICE = torch.device("cuda", 0)
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _linear(m, k, n, group=128, act="none", bias=True, out="bf16"):
    return {"kind": "linear", "m": m, "k": k, "n": n, "group": group, "act": act, "bias": bias, "out": out}


def _sage(b, hq, hkv, lq, lk, d, layout="HND", causal=False):
    return {"kind": "sage", "b": b, "hq": hq, "hkv": hkv, "lq": lq, "lk": lk, "d": d, "layout": layout,
            "causal": causal}


def _w8a8(b, hq, hkv, lq, lk, d, dtype="bf16", causal=False):
    return {"kind": "w8a8", "b": b, "hq": hq, "hkv": hkv, "lq": lq, "lk": lk, "d": d, "dtype": dtype,
            "causal": causal}


def _block(dim, heads, ffn, f, h, w, text):
    return {"kind": "block", "dim": dim, "heads": heads, "ffn": ffn, "f": f, "h": h, "w": w, "text": text}


def listed():
    return [
        # Wan 1.3B's time projection of one prompt: one row, launches and latency only.
        dict(_linear(1, 1536, 9216), name="linear_row"),
        # Cross-attention's fused k / v projection of the 512 text tokens (Wan 14B).
        dict(_linear(512, 5120, 10240), name="linear_text"),
        # An ordinary projection: 4096 tokens through Wan 1.3B's FFN up layer.
        dict(_linear(4096, 1536, 8960), name="linear_4096"),
        # A SwiGLU model's FFN down layer on the reference's group of 256, ragged rows, fp16 output.
        dict(_linear(2050, 14336, 5376, group=256, act="swiglu", bias=False, out="f16"), name="linear_swiglu_f16"),
        # The largest linear: a whole 480p video's FFN down layer (Wan 14B) with its GELU.
        dict(_linear(32760, 13824, 5120, act="gelu_tanh"), name="linear_gelu_32760"),
        # Grouped-query attention over a short prompt, head_dim 64, the NHD layout ComfyUI hands over.
        dict(_sage(2, 8, 2, 257, 300, 64, layout="NHD"), name="sage_short_gqa"),
        # Causal grouped-query attention at an ordinary odd length.
        dict(_sage(2, 16, 4, 4001, 4001, 128, layout="NHD", causal=True), name="sage_causal_gqa"),
        # Wan 1.3B self-attention on a short clip.
        dict(_sage(1, 12, 12, 8190, 8190, 128), name="sage_8190"),
        # Wan 14B self-attention on a whole 480p video: the largest call.
        dict(_sage(1, 40, 40, 32760, 32760, 128), name="sage_32760"),
        # W8A8 attention (the loader's default backend) over one 480p frame of Wan 1.3B.
        dict(_w8a8(1, 12, 12, 1560, 1560, 128), name="w8a8_1560"),
        # W8A8 attention at the reference's published 56 heads x 4096 tokens, fp16 as its A40 ran it.
        dict(_w8a8(1, 56, 56, 4096, 4096, 128, dtype="f16"), name="w8a8_4096_f16"),
        # One whole Wan 1.3B block on a 17-frame 480p clip (5 x 30 x 52 latents): norms, modulation, RoPE, both
        # attentions, the seven projections and the residual adds.
        dict(_block(1536, 12, 8960, 5, 30, 52, 512), name="wan_block_7800"),
    ]


def _log(rng, low, high):
    """An integer spread over the logarithm of [low, high]."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["sage"] * 4 + ["w8a8"] * 2 + ["block"])
    if kind == "linear":
        group = rng.choice([128, 128, 256])
        k = group * _log(rng, 512 // group, 14336 // group)
        n = 8 * _log(rng, 32, 2688)
        m = _log(rng, 1, max(1, min(32760, int(4.6e12 / (2 * k * n)))))
        return _linear(m, k, n, group, rng.choice(["none", "none", "gelu_tanh", "swiglu"]), rng.random() < 0.7,
                       rng.choice(["bf16", "bf16", "bf16", "f16", "f32"]))
    if kind == "block":
        dim, heads, ffn = rng.choice([(1536, 12, 8960), (1536, 12, 8960), (5120, 40, 13824)])
        h, w = rng.choice([(30, 52), (30, 52), (32, 32), (45, 80), (26, 38)])
        f = _log(rng, 1, max(1, min(21, (16380 if dim == 5120 else 32760) // (h * w))))
        return _block(dim, heads, ffn, f, h, w, rng.choice([512, 512, rng.randint(77, 511)]))
    d = rng.choice([64, 128, 128, 128])
    hkv, rep = rng.choice([(_log(rng, 1, 40), 1), (_log(rng, 1, 40), 1), (_log(rng, 1, 8), rng.choice([2, 4]))])
    b = rng.choice([1, 1, 1, 2])
    causal, cross = False, rng.random() < 0.3
    most = 2.1e13 if kind == "sage" else 8e12
    lk = _log(rng, 16, 512) if cross else 0
    per = 4.0 * b * hkv * rep * d
    lq = _log(rng, 64, 32760)
    while per * lq * (lk or lq) > most or 8.0 * b * hkv * rep * d * lq > 3e9:
        lq = int(lq * 0.8)
    if not cross:
        lk, causal = lq, rng.random() < 0.25
    if kind == "sage":
        return _sage(b, hkv * rep, hkv, lq, lk, d, rng.choice(["HND", "NHD"]), causal)
    return _w8a8(b, hkv * rep, hkv, lq, lk, d, rng.choice(["bf16", "f16"]), causal)


def _tokens(case):
    return case["f"] * case["h"] * case["w"]


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEVICE)


def _attention_inputs(case, seed, dtype):
    """Q, K, V with unit-variance channels; K carries the per-head channel offset that smoothing is there for."""
    g = _generator(seed)
    b, hq, hkv, lq, lk, d = (case[x] for x in ("b", "hq", "hkv", "lq", "lk", "d"))
    q = _randn(g, b, hq, lq, d).to(dtype)
    k = (_randn(g, b, hkv, lk, d) + 2.0 * _randn(g, b, hkv, 1, d)).to(dtype)
    v = _randn(g, b, hkv, lk, d).to(dtype)
    return q, k, v


def _linear_inputs(case, seed):
    """Activations with 0.1 % outlier channels (x20), full-range int8 weight codes, per-channel scales."""
    g = _generator(seed)
    width = case["k"] * (2 if case["act"] == "swiglu" else 1)
    x = _randn(g, case["m"], width)
    x[:, torch.randperm(width, generator=g, device=DEVICE)[: max(1, round(0.001 * width))]] *= 20.0
    w = torch.randint(-127, 128, (case["n"], case["k"]), generator=g, device=DEVICE, dtype=torch.int8)
    ws = 1e-3 + 4e-3 * torch.rand(case["n"], generator=g, device=DEVICE)
    bias = 0.02 * _randn(g, case["n"]) if case["bias"] else None
    return x.to(torch.bfloat16), w, ws, bias


def _block_inputs(case, seed):
    cfg = wan_block.WanBlockConfig(dim=case["dim"], heads=case["heads"], ffn_dim=case["ffn"])
    block, _ = wan_block.random_block(cfg, seed, DEVICE)
    g = _generator(seed + 1)
    x = _randn(g, 1, _tokens(case), case["dim"]).to(torch.bfloat16)
    e = 0.1 * _randn(g, 1, 6, case["dim"])
    context = _randn(g, 1, case["text"], case["dim"]).to(torch.bfloat16)
    return block, x, e, context, wan_block.rope_freqs((case["f"], case["h"], case["w"]), 128, device=DEVICE)


def prepare(case, seed):
    if case["kind"] == "linear":
        inputs = _linear_inputs(case, seed)
    elif case["kind"] == "block":
        inputs = _block_inputs(case, seed)
    elif case["kind"] == "sage":
        inputs = _attention_inputs(case, seed, torch.bfloat16)
        if case["layout"] == "NHD":
            inputs = tuple(t.transpose(1, 2).contiguous() for t in inputs)
    else:
        inputs = _attention_inputs(case, seed, DTYPES[case["dtype"]])
    return case, inputs


def run(state):
    case, inputs = state
    if case["kind"] == "linear":
        x, w, ws, bias = inputs
        return integration.int8_linear(x, w, ws, bias, out_dtype=DTYPES[case["out"]], convrot=True,
                                       convrot_groupsize=case["group"], input_act=case["act"])
    if case["kind"] == "sage":
        return turing_sage.sageattn(*inputs, tensor_layout=case["layout"], is_causal=case["causal"])
    if case["kind"] == "w8a8":
        return turing_sage.w8a8attn(*inputs, is_causal=case["causal"])
    block, x, e, context, freqs = inputs
    return block(x, e, context, freqs)


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        width = k * (2 if case["act"] == "swiglu" else 1)
        return {"bytes": 2 * m * width + n * k + 8 * n + (4 if case["out"] == "f32" else 2) * m * n,
                "flops": 2.0 * m * n * k}
    if case["kind"] == "block":
        c, f, l, t = case["dim"], case["ffn"], _tokens(case), case["text"]
        weights = c * (3 * c + c + c + 2 * c + c + 2 * f)
        return {"bytes": weights + 4 * l * c + 2 * t * c + 4 * l * 128 * 2,
                "flops": 2.0 * l * c * (6 * c + 2 * f) + 4.0 * t * c * c + 4.0 * c * l * (l + t)}
    b, hq, hkv, lq, lk, d = (case[x] for x in ("b", "hq", "hkv", "lq", "lk", "d"))
    pairs = lq * (lq + 1) / 2 if case["causal"] else lq * lk
    return {"bytes": 4 * b * d * (hq * lq + hkv * lk), "flops": 4.0 * b * hq * d * pairs}


def tolerance(case):
    if case["kind"] == "linear":
        # codes and accumulators are whole numbers: one rounding to the output type, and now and then a code that
        # another order of the rotation's 32-bit sums puts on the other side of a tie
        return {"rel": 6e-3}
    if case["kind"] == "sage":
        return {"rel": 1e-2}  # probabilities and outputs in bf16
    if case["kind"] == "w8a8":
        return {"rel": 1.5e-2}  # probabilities in 8 bits below their row's running maximum
    return {"rel": 1e-2}  # bf16 residual stream through three sublayers


# -- 64-bit results ------------------------------------------------------------


def _rotation(group):
    """ConvRot's orthogonal matrix: Kronecker powers of the regular 4 x 4 Hadamard matrix, for 128 with a 2 x 2 one."""
    r4 = 0.5 * torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64)
    r2 = math.sqrt(0.5) * torch.tensor([[1, 1], [1, -1]], dtype=torch.float64)
    m = torch.kron(r4 if group == 256 else r2, torch.kron(r4, torch.kron(r4, r4)))
    return m.to(DEVICE)


def _rotate(x, group):
    return (x.reshape(-1, group) @ _rotation(group).T).reshape(x.shape)


def _exact_linear(case, seed):
    """The quantized linear with the rounding points of its definition (bf16 rotated rows and quotients)."""
    x, w, ws, bias = _linear_inputs(case, seed)
    w64 = w.double().T.contiguous()
    out = []
    for rows in x.split(2048):
        a = rows.double()
        if case["act"] == "gelu_tanh":
            a = torch.nn.functional.gelu(a, approximate="tanh").to(torch.bfloat16).double()
        elif case["act"] == "swiglu":
            gate, up = a.chunk(2, -1)
            a = gate * torch.sigmoid(gate) * up
        y = _rotate(a, case["group"])
        scale = y.abs().amax(-1, keepdim=True) / 127
        codes = (y.to(torch.bfloat16).double() / scale.to(torch.bfloat16).double()).to(torch.bfloat16)
        codes = codes.double().round().clamp(-128, 127)
        y = (codes @ w64) * scale * ws.double()
        out.append(y + bias.double() if bias is not None else y)
    return torch.cat(out)


def _softmax_attention(q, k, v, causal, scale):
    """Attention of one head in 64 bits, in slices of queries."""
    out = []
    for start in range(0, q.shape[0], 4096):
        s = (q[start:start + 4096] @ k.T) * scale
        if causal:
            rows = torch.arange(start, start + s.shape[0], device=s.device)[:, None]
            s = s.masked_fill(torch.arange(k.shape[0], device=s.device)[None] > rows, -math.inf)
        out.append(torch.softmax(s, -1) @ v)
    return torch.cat(out)


def _block_codes(x, block=128):
    """x [L, D] as its symmetric 8-bit codes times their scales, one scale for each `block` tokens."""
    length = x.shape[0]
    t = torch.nn.functional.pad(x, (0, 0, 0, -length % block)).reshape(-1, block, x.shape[1])
    scale = t.abs().amax((1, 2), keepdim=True).clamp(min=1e-7) / 127
    return ((t / scale).round().clamp(-128, 127) * scale).reshape(-1, x.shape[1])[:length]


def _exact_attention(case, seed):
    quantized = case["kind"] == "sage"  # W8A8 rotates Q and K first: its result is set against plain attention
    q, k, v = _attention_inputs(case, seed, torch.bfloat16 if quantized else DTYPES[case["dtype"]])
    rep = case["hq"] // case["hkv"]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    for b in range(case["b"]):
        for h in range(case["hkv"]):
            kh, vh = k[b, h].double(), v[b, h].double()
            if quantized:
                kh = _block_codes(kh - kh.mean(0, keepdim=True).to(torch.bfloat16).double())
            for r in range(h * rep, (h + 1) * rep):
                qh = q[b, r].double()
                qh = _block_codes(qh) if quantized else qh
                out[b, r] = _softmax_attention(qh, kh, vh, case["causal"], case["d"] ** -0.5)
    return out.transpose(1, 2) if case.get("layout") == "NHD" else out


def _exact_block(case, seed):
    """The block on its 8-bit weights and the bf16 rotary table, with nothing else quantized or rounded."""
    block, x, e, context, freqs = _block_inputs(case, seed)
    heads, d = case["heads"], case["dim"] // case["heads"]
    eps = block.cfg.eps
    x, context = x[0].double(), context[0].double()
    rot = freqs[0, :, 0].to(torch.bfloat16).double()  # [L, D/2, 2, 2]
    mod = (block.modulation + e)[0].to(torch.bfloat16).double()

    def lin(layer, a):
        return (_rotate(a, layer.group) @ layer.weight.double().T) * layer.weight_scale.double() + layer.bias.double()

    def norm(a):
        return torch.nn.functional.layer_norm(a, (a.shape[-1],), eps=eps)

    def rms(a, weight):
        return a * torch.rsqrt(a.square().mean(-1, keepdim=True) + eps) * weight.double()

    def rope(a):
        pairs = a.reshape(-1, heads, d // 2, 2)
        return torch.stack([(rot[:, None, :, i] * pairs).sum(-1) for i in (0, 1)], -1).reshape(a.shape)

    def attention(q, k, v):
        q, k, v = (t.reshape(-1, heads, d) for t in (q, k, v))
        return torch.cat([_softmax_attention(q[:, h], k[:, h], v[:, h], False, d ** -0.5) for h in range(heads)], -1)

    q, k, v = lin(block.self_qkv, norm(x) * (1 + mod[1]) + mod[0]).chunk(3, -1)
    a = attention(rope(rms(q, block.self_norm_q)), rope(rms(k, block.self_norm_k)), v)
    x = x + lin(block.self_o, a) * mod[2]
    q = lin(block.cross_q, norm(x) * block.norm3_weight.double() + block.norm3_bias.double())
    k, v = lin(block.cross_kv, context).chunk(2, -1)
    x = x + lin(block.cross_o, attention(rms(q, block.cross_norm_q), rms(k, block.cross_norm_k), v))
    a = lin(block.ffn_up, norm(x) * (1 + mod[4]) + mod[3])
    x = x + lin(block.ffn_down, torch.nn.functional.gelu(a, approximate="tanh")) * mod[5]
    return x[None]


def exact(case, seed):
    if case["kind"] == "linear":
        return _exact_linear(case, seed)
    return _exact_block(case, seed) if case["kind"] == "block" else _exact_attention(case, seed)
