"""The work a user of this framework has it do, as measurable cases.

Two kinds of callers stand behind them:

* a serving engine that holds one decoder behind the ModelForward boundary
  (``HipForward``): it clears the cache, restores a cached prefix or prefills
  a prompt in chunks, then decodes token by token and reads the logits of
  every forward;
* a backend that calls the op-level C entry points on device buffers of its
  own: one projection (GEMV for a token, GEMM for a chunk) or one attention
  layer over the paged K/V cache.

``listed()`` names twelve cases from the smallest call to the largest;
``draw()`` gives more of the same ranges. A case is plain values; its "kind"
picks the entry point. Shapes are those of the decoders in
``cheetah_amd.configs`` (all layers of Qwen2-0.5B; two layers of the large
ones with a 32,000-token vocabulary, so that a case stays a block of layers
and not a copy of the whole checkpoint) or generic sizes.
"""
import ctypes
import math

import numpy as np
import torch

from cheetah_amd import configs, hip

FMT_LIMIT = {"q8": 127, "q4": 7}
# (q heads, KV heads, head dim) of the decoders served.
HEADS = ((14, 2, 64), (32, 8, 128), (28, 4, 128))
# (rows, cols) of the decoders' projections: qkv, o, gate/up, down.
PROJ = ((1152, 896), (896, 896), (4864, 896), (896, 4864),
        (6144, 4096), (4096, 4096), (14336, 4096), (4096, 14336),
        (4608, 3584), (3584, 3584), (18944, 3584), (3584, 18944))
HEAD_MATS = ((151936, 896), (32000, 4096), (128256, 4096))
PAGE = 64
MODELS = {
    "qwen2-0.5b": configs.QWEN2_0_5B,
    "llama3-8b/2": configs.LLAMA3_8B.replace(name="llama3-8b/2", num_layers=2, vocab_size=32000),
    "qwen2-7b/2": configs.QWEN2_7B.replace(name="qwen2-7b/2", num_layers=2, vocab_size=32000),
}
GEMM_MAX = 18944 * 3584 * 1024


def listed():
    return [
        # One token through the smallest projection: the launch is most of it.
        {"name": "gemv_bf16_qkv_0.5b", "kind": "gemv", "fmt": "bf16", "rows": 1152, "cols": 896},
        # The quantized decode step's long-K projection.
        {"name": "gemv_q4_down_8b", "kind": "gemv", "fmt": "q4", "rows": 4096, "cols": 14336},
        # The largest matrix a decode step streams: a BF16 LM head.
        {"name": "gemv_bf16_head", "kind": "gemv", "fmt": "bf16", "rows": 128256, "cols": 4096},
        # The ragged remainder of a prompt through a Q8 projection.
        {"name": "gemm_q8_ragged", "kind": "gemm", "fmt": "q8", "rows": 4096, "cols": 4096, "n": 389},
        # A 512-row chunk of a Q4 decoder through gate (or up).
        {"name": "gemm_q4_gate_8b", "kind": "gemm", "fmt": "q4", "rows": 14336, "cols": 4096, "n": 512},
        # A 1,024-row chunk of a BF16 decoder through gate: the largest GEMM.
        {"name": "gemm_bf16_gate_7b", "kind": "gemm", "fmt": "bf16", "rows": 18944, "cols": 3584, "n": 1024},
        # One decoded token over a short, ragged context.
        {"name": "attn_decode_577", "kind": "attn", "q_heads": 14, "kv_heads": 2, "hd": 64, "rows": 1, "offset": 576},
        # One decoded token over a long context.
        {"name": "attn_decode_16k", "kind": "attn", "q_heads": 32, "kv_heads": 8, "hd": 128, "rows": 1,
         "offset": 16383},
        # A prefill chunk late in a long prompt.
        {"name": "attn_prefill_512_on_4k", "kind": "attn", "q_heads": 32, "kv_heads": 8, "hd": 128, "rows": 512,
         "offset": 4096},
        # Token-by-token decode after a restored prefix, logits read each step.
        {"name": "decode_qwen2_0.5b", "kind": "decode", "model": "qwen2-0.5b", "quant": "bf16", "kv": "bf16",
         "ctx": 512, "steps": 16},
        # A short prompt through the whole small decoder.
        {"name": "prefill_qwen2_0.5b", "kind": "prefill", "model": "qwen2-0.5b", "quant": "bf16", "kv": "bf16",
         "n": 512, "chunk": 128},
        # A prompt through quantized layers with the exact (f32) K/V cache.
        {"name": "prefill_8b_layers_f32kv", "kind": "prefill", "model": "llama3-8b/2", "quant": "q4", "kv": "f32",
         "n": 1500, "chunk": 512},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _matrix(rng):
    """A projection of the decoders, or a generic size (some of them odd)."""
    if rng.random() < 0.55:
        return rng.choice(PROJ)
    rows, cols = _log_int(rng, 64, 20000), _log_int(rng, 128, 16000)
    if rng.random() < 0.5:
        rows, cols = max(64, rows // 64 * 64), max(128, cols // 64 * 64)
    return rows, cols


def draw(rng):
    kind = rng.choice(("gemv", "gemv", "gemm", "gemm", "gemm", "attn_decode", "attn_prefill", "decode", "prefill",
                       "prefill"))
    if kind == "gemv":
        rows, cols = rng.choice(HEAD_MATS[:2]) if rng.random() < 0.15 else _matrix(rng)
        return {"kind": "gemv", "fmt": rng.choice(("bf16", "q8", "q4")), "rows": rows, "cols": cols}
    if kind == "gemm":
        rows, cols = _matrix(rng)
        n = max(2, min(_log_int(rng, 2, 2048), GEMM_MAX // (rows * cols)))
        return {"kind": "gemm", "fmt": rng.choice(("bf16", "q8", "q4")), "rows": rows, "cols": cols, "n": n}
    if kind.startswith("attn"):
        qh, kvh, hd = rng.choice(HEADS)
        if kind == "attn_decode":
            rows, offset = 1, _log_int(rng, 16, 32768) - 1
        else:
            rows, offset = _log_int(rng, 16, 1024), rng.choice((0, _log_int(rng, 64, 4096)))
        return {"kind": "attn", "q_heads": qh, "kv_heads": kvh, "hd": hd, "rows": rows, "offset": offset}
    model = rng.choice(tuple(MODELS))
    quant = "bf16" if model == "qwen2-7b/2" else rng.choice(("bf16", "q8", "q4"))
    case = {"kind": kind, "model": model, "quant": quant, "kv": rng.choice(("bf16", "f32"))}
    if kind == "decode":
        case.update(ctx=_log_int(rng, 32, 1024), steps=rng.choice((4, 8, 16)))
    else:
        case.update(n=_log_int(rng, 32, 1500), chunk=rng.choice((128, 256, 512)))
    return case


# ---------------------------------------------------------------------------
# Inputs, made on the GPU from the seed alone.
# ---------------------------------------------------------------------------

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + salt)
    return g


class _Buf:
    """A framework device buffer that torch can fill and read in place."""

    def __init__(self, tensor):
        tensor = tensor.contiguous()
        self.buf = hip.DeviceBuffer(max(tensor.numel() * tensor.element_size(), 4))
        kind = {torch.float32: "<f4", torch.uint8: "|u1", torch.int16: "<i2", torch.int32: "<i4"}[tensor.dtype]
        self.__cuda_array_interface__ = {"shape": tuple(tensor.shape), "typestr": kind, "version": 2,
                                         "data": (int(self.buf.ptr), False), "strides": None}
        self.view = torch.as_tensor(self, device="cuda")
        self.view.copy_(tensor)

    @property
    def ptr(self):
        return self.buf.ptr


def _bf16_weight(g, rows, cols):
    return (torch.randn(rows, cols, generator=g, device="cuda") * 0.02).to(torch.bfloat16)


def _weight(fmt, rows, cols, g):
    """(buffer in the framework's weight layout, its values as (codes, scales))."""
    if fmt == "bf16":
        w = _bf16_weight(g, rows, cols)
        return w.view(torch.int16), (w, None)
    limit = FMT_LIMIT[fmt]
    codes = torch.randn(rows, cols, generator=g, device="cuda").mul_(limit / 4).round_().clamp_(-limit, limit)
    codes = codes.to(torch.int8)
    scales = torch.rand(rows, generator=g, device="cuda") * 0.001 + 0.08 / limit
    stride = (hip.buffer_bytes(fmt, rows, cols) - 4 * rows) // rows
    pay = torch.zeros(rows, stride, dtype=torch.uint8, device="cuda")
    if fmt == "q8":
        pay[:, :cols] = codes.view(torch.uint8)
    else:
        nib = codes.view(torch.uint8) & 0xF
        pay[:, :(cols + 1) // 2] = nib[:, 0::2]
        pay[:, :cols // 2] |= nib[:, 1::2] << 4
    return torch.cat([scales.view(torch.uint8), pay.reshape(-1)]), (codes, scales)


def _attn_inputs(case, seed):
    qh, kvh, hd, rows, offset = (case[k] for k in ("q_heads", "kv_heads", "hd", "rows", "offset"))
    g = _gen(seed)
    ctx = offset + rows
    pages = -(-ctx // PAGE)
    q = torch.randn(rows, qh * hd, generator=g, device="cuda")
    k = torch.randn(pages * PAGE, kvh, hd, generator=g, device="cuda").to(torch.bfloat16)
    v = torch.randn(pages * PAGE, kvh, hd, generator=g, device="cuda").to(torch.bfloat16)
    table = torch.randperm(pages, generator=g, device="cuda").to(torch.int32)
    return q, k, v, table, pages


def _model_weights(shape, seed):
    """Unit id -> BF16 tensor on the GPU."""
    g = _gen(seed)
    w = {"model.embed_tokens.weight": _bf16_weight(g, shape.vocab_size, shape.hidden_size)}

    def gain():
        return (1 + 0.1 * torch.randn(shape.hidden_size, generator=g, device="cuda")).to(torch.bfloat16)

    for layer in range(shape.num_layers):
        p = f"model.layers.{layer}."
        w[p + "input_layernorm.weight"] = gain()
        w[p + "post_attention_layernorm.weight"] = gain()
        for unit, rows, cols in shape.linear_units(layer):
            w[unit] = _bf16_weight(g, rows, cols)
        if shape.qkv_bias:
            for name, n in (("q", shape.q_dim), ("k", shape.kv_dim), ("v", shape.kv_dim)):
                w[p + f"self_attn.{name}_proj.bias"] = _bf16_weight(g, 1, n).reshape(n)
    w["model.norm.weight"] = gain()
    if not shape.tie_word_embeddings:
        w["lm_head.weight"] = _bf16_weight(g, shape.vocab_size, shape.hidden_size)
    return w


def _tokens(case, shape, seed):
    n = case["ctx"] + case["steps"] if case["kind"] == "decode" else case["n"]
    return torch.randint(0, shape.vocab_size, (n,), generator=_gen(seed, 1), device="cuda").cpu().numpy().astype(np.uint32)


def _op(case):
    return getattr(hip.lib(), f"cheetah_hip_{case['kind']}_{case['fmt']}")


def prepare(case, seed):
    hip.init(0)
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        rows, cols, n = case["rows"], case["cols"], case.get("n", 1)
        g = _gen(seed)
        w, _ = _weight(case["fmt"], rows, cols, g)
        x = torch.randn(n, cols, generator=g, device="cuda")
        y = torch.zeros((n, rows) if kind == "gemm" else (rows,), device="cuda")
        w, x, y = _Buf(w), _Buf(x), _Buf(y)
        torch.cuda.synchronize()
        args = (w.ptr, rows, cols, x.ptr, y.ptr) if kind == "gemv" else (w.ptr, rows, cols, x.ptr, n, y.ptr)
        return {"call": _op(case), "args": args, "out": y.view, "keep": (w, x, y)}
    if kind == "attn":
        qh, kvh, hd, rows, offset = (case[k] for k in ("q_heads", "kv_heads", "hd", "rows", "offset"))
        q, k, v, table, pages = _attn_inputs(case, seed)

        def paged(t):
            p = torch.empty(pages, kvh, PAGE, hd, dtype=torch.bfloat16, device="cuda")
            p[table.long()] = t.view(pages, PAGE, kvh, hd).transpose(1, 2)
            return p.view(torch.int16)

        q, k, v, table = _Buf(q), _Buf(paged(k)), _Buf(paged(v)), _Buf(table)
        out = _Buf(torch.zeros(rows, qh * hd, device="cuda"))
        torch.cuda.synchronize()
        view = hip.KvView(k.ptr, v.ptr, table.ptr, PAGE, kvh, hd)
        args = (q.ptr, ctypes.byref(view), qh, rows, offset, out.ptr)
        return {"call": hip.lib().cheetah_hip_attention, "args": args, "out": out.view,
                "keep": (q, k, v, table, out, view)}
    shape = MODELS[case["model"]]
    weights = {k: t.cpu().view(torch.int16).numpy().view(np.uint16) for k, t in _model_weights(shape, seed).items()}
    tokens = _tokens(case, shape, seed)
    # The pages of the prompt, a second run's own pages and a copied one.
    g = hip.HipForward(shape, weights, quant=None if case["quant"] == "bf16" else case["quant"], kv=case["kv"],
                       kv_capacity=len(tokens) + 3 * PAGE, max_chunk_rows=case.get("chunk", 256))
    state = {"model": g, "tokens": tokens}
    if kind == "decode":
        g.forward(tokens[:case["ctx"]], 0, chunk_rows=256)
        state.update(snapshot=g.kv_snapshot(), ctx=case["ctx"])
    else:
        state["chunk"] = case["chunk"]
    return state


def run(state):
    if "call" in state:
        hip.check(state["call"](*state["args"]))
        return state["out"]
    g, tokens = state["model"], state["tokens"]
    g.clear_cache()
    if "snapshot" not in state:
        return g.forward(tokens, 0, chunk_rows=state["chunk"])
    ctx = state["ctx"]
    g.restore_kv_prefix(state["snapshot"], ctx)
    return [g.forward(tokens[i:i + 1], i) for i in range(ctx, len(tokens))]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how far another implementation may be.
# ---------------------------------------------------------------------------

def _matrix_bytes(fmt, rows, cols):
    return {"bf16": 2 * rows * cols, "q8": rows * cols + 4 * rows, "q4": rows * cols / 2 + 4 * rows}[fmt]


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        rows, cols, n = case["rows"], case["cols"], case.get("n", 1)
        return {"bytes": _matrix_bytes(case["fmt"], rows, cols) + 4 * n * (rows + cols), "flops": 2 * rows * cols * n}
    if kind == "attn":
        qh, kvh, hd, rows, offset = (case[k] for k in ("q_heads", "kv_heads", "hd", "rows", "offset"))
        keys = rows * offset + rows * (rows + 1) / 2
        return {"bytes": 2 * 2 * (offset + rows) * kvh * hd + 2 * 4 * rows * qh * hd, "flops": 4 * qh * hd * keys}
    shape = MODELS[case["model"]]
    linear = sum(_matrix_bytes(case["quant"], r, c) for i in range(shape.num_layers) for _, r, c in shape.linear_units(i))
    head = 2 * shape.head_params()
    kv_row = 2 * shape.kv_dim * (4 if case["kv"] == "f32" else 2) * shape.num_layers
    if kind == "decode":
        ctx, steps = case["ctx"], case["steps"]
        keys = steps * ctx + steps * (steps + 1) / 2
        return {"bytes": steps * (linear + head + 4 * shape.vocab_size) + keys * kv_row,
                "flops": 2 * steps * (shape.linear_params() + shape.head_params())
                + 4 * shape.q_dim * keys * shape.num_layers}
    n = case["n"]
    return {"bytes": linear + head + 4 * shape.vocab_size + 2 * n * shape.hidden_size + n * kv_row,
            "flops": 2 * n * shape.linear_params() + 2 * shape.head_params()
            + 4 * shape.q_dim * n * (n + 1) / 2 * shape.num_layers}


def tolerance(case):
    """About four times the distance from ``exact`` seen over the ranges (GEMV
    2.5e-7; GEMM 2.7e-6 and attention 3.5e-6, whose f32 activations, queries
    and probabilities are two BF16 halves on the matrix cores; whole calls
    3.7e-5 on an f32 cache and 4.2e-4 on a BF16 one, where the last bit of a
    rounded K or V may fall the other way)."""
    kind = case["kind"]
    if kind == "gemv":
        return {"rel": 1e-6}
    if kind == "gemm":
        return {"rel": 1.2e-5}
    if kind == "attn":
        return {"rel": 1.5e-5}
    return {"rel": 1.5e-4 if case["kv"] == "f32" else 1.7e-3}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch.
# ---------------------------------------------------------------------------

def _quantized(w, quant):
    """A BF16 matrix's values after row-wise quantization, as the layout
    defines it: scale = max|w| / limit in f32 (1 for a zero row), codes
    w / scale in f32 rounded half away from zero. (Divided in 64 bits and
    rounded to f32: torch divides by a number as a product on the GPU.)"""
    w = w.double()
    if quant == "bf16":
        return w
    limit = FMT_LIMIT[quant]
    scale = (w.abs().amax(dim=1, keepdim=True) / limit).float().double()
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    q = (w / scale).float().double()
    return (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp_(-limit, limit) * scale


def _attention64(q, k, v, offset):
    """q [rows, heads, hd], k/v [ctx, kv_heads, hd]; causal from `offset`."""
    rows, qh, hd = q.shape
    group = qh // k.shape[1]
    last = torch.arange(offset, offset + rows, device="cuda")[:, None]
    mask = torch.arange(k.shape[0], device="cuda")[None, :] > last
    out = torch.empty_like(q)
    for h in range(qh):
        s = q[:, h] @ k[:, h // group].t().contiguous() / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill_(mask, -math.inf), dim=1) @ v[:, h // group].contiguous()
    return out


def _rope64(x, shape, cos, sin):
    half = shape.rotary_dim // 2
    a, b, rest = x[..., :half], x[..., half:2 * half], x[..., 2 * half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, rest], dim=-1)


def _model64(case, seed):
    shape = MODELS[case["model"]]
    w = _model_weights(shape, seed)
    ids = torch.from_numpy(_tokens(case, shape, seed).astype(np.int64)).cuda()
    # The rotation's angles are f32 by definition: pos * theta^(-2i/d).
    half = shape.rotary_dim // 2
    freq = np.power(np.float32(shape.rope_theta), (np.float32(-2) * np.arange(half, dtype=np.float32)
                                                   / np.float32(shape.rotary_dim))).astype(np.float32)
    angle = np.arange(len(ids), dtype=np.float32)[:, None] * freq[None, :]
    cos, sin = (torch.from_numpy(f(angle).astype(np.float32)).cuda().double()[:, None, :] for f in (np.cos, np.sin))
    x = w["model.embed_tokens.weight"][ids].double()

    def norm(t, unit):
        return t * torch.rsqrt((t * t).mean(dim=-1, keepdim=True) + shape.rms_eps) * w[unit].double()

    def linear(t, unit):
        y = t @ _quantized(w[unit + ".weight"], case["quant"]).t().contiguous()
        bias = w.get(unit + ".bias")
        return y if bias is None else y + bias.double()

    for layer in range(shape.num_layers):
        p = f"model.layers.{layer}."
        t = norm(x, p + "input_layernorm.weight")
        q, k, v = (linear(t, p + f"self_attn.{c}_proj").view(len(ids), -1, shape.head_dim) for c in "qkv")
        q, k = _rope64(q, shape, cos, sin), _rope64(k, shape, cos, sin)
        if case["kv"] == "bf16":  # the cache's element type is part of the result
            k, v = k.float().to(torch.bfloat16).double(), v.float().to(torch.bfloat16).double()
        x = x + linear(_attention64(q, k, v, 0).reshape(len(ids), -1), p + "self_attn.o_proj")
        t = norm(x, p + "post_attention_layernorm.weight")
        x = x + linear(torch.nn.functional.silu(linear(t, p + "mlp.gate_proj")) * linear(t, p + "mlp.up_proj"),
                       p + "mlp.down_proj")
    x = norm(x[case.get("ctx", len(ids) - 1):], "model.norm.weight")
    head = w["model.embed_tokens.weight" if shape.tie_word_embeddings else "lm_head.weight"]
    logits = torch.cat([x @ part.double().t().contiguous() for part in head.split(16384)], dim=1)
    return list(logits.cpu().numpy()) if case["kind"] == "decode" else logits[0].cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        rows, cols, n = case["rows"], case["cols"], case.get("n", 1)
        g = _gen(seed)
        _, (codes, scales) = _weight(case["fmt"], rows, cols, g)
        x = torch.randn(n, cols, generator=g, device="cuda").double()
        y = torch.cat([x @ part.double().t().contiguous() for part in codes.split(16384)], dim=1)
        if scales is not None:
            y = y * scales.double()
        return y if kind == "gemm" else y[0]
    if kind == "attn":
        q, k, v, _, _ = _attn_inputs(case, seed)
        rows, offset, hd = case["rows"], case["offset"], case["hd"]
        ctx = offset + rows
        out = _attention64(q.view(rows, -1, hd).double(), k[:ctx].double(), v[:ctx].double(), offset)
        return out.reshape(rows, -1)
    return _model64(case, seed)
