"""Forward-level parity of the HIP ModelForward against the CPU oracle.

Bars (north star): logits within 1e-2 relative of the reference path
(f32 accumulation; the device keeps K/V in BF16 where the reference keeps
f32), greedy token sequences identical for the first 32 decode steps.
Device invariants from the reference's decoder tests (decoder.rs:1710-1818):
KV continuation and snapshot -> restore -> continue are bit-exact.
"""
import json
import os

import numpy as np
import pytest

import golden_checks
from cheetah_amd import configs, synth

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


@pytest.fixture(scope="module")
def hip():
    from cheetah_amd import hip as h
    h.init(0)
    return h


def rel_err(got, ref):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    return float(np.max(np.abs(got - ref)) / max(np.max(np.abs(ref)), 1e-30))


def bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


_WEIGHTS = {}


def weights(shape):
    if shape.name not in _WEIGHTS:
        _WEIGHTS.clear()
        _WEIGHTS[shape.name] = synth.make_weights(shape)
    return _WEIGHTS[shape.name]


TINY = [configs.TINY_QWEN2, configs.TINY_LLAMA]


@pytest.mark.parametrize("kv", ["bf16", "f32"])
@pytest.mark.parametrize("quant", [None, "q8", "q4"])
@pytest.mark.parametrize("shape", TINY, ids=lambda s: s.name)
def test_tiny_forward_matches_oracle(hip, oracle, shape, quant, kv):
    """Logits of chunked prefill and of decode steps. The oracle with the
    device's KV precision isolates kernel arithmetic (tight bound); the
    reference semantics (f32 KV) are held to the 1e-2 bar."""
    w = weights(shape)
    g = hip.HipForward(shape, w, quant=quant, kv_capacity=512, max_chunk_rows=64, kv=kv)
    r_same = oracle.RefModel(shape, w, quant=quant, kv_bf16=(kv == "bf16"))
    r_ref = oracle.RefModel(shape, w, quant=quant)
    toks = synth.make_tokens(shape.vocab_size, 60, seed=2)
    lg = g.forward(toks[:45], 0, chunk_rows=16)
    ls = r_same.forward(toks[:45], 0, chunk_rows=16)
    lr = r_ref.forward(toks[:45], 0, chunk_rows=16)
    assert rel_err(lg, ls) < 1e-3
    assert rel_err(lg, lr) < 1e-2
    for i in range(45, 60):
        lg = g.forward(toks[i:i + 1], i)
        ls = r_same.forward(toks[i:i + 1], i)
        lr = r_ref.forward(toks[i:i + 1], i)
        assert rel_err(lg, ls) < 1e-3, i
        assert rel_err(lg, lr) < 1e-2, i
    assert g.kv_len() == 60


@pytest.mark.parametrize("kv", ["bf16", "f32"])
@pytest.mark.parametrize("shape", TINY, ids=lambda s: s.name)
def test_tiny_greedy_32_steps_token_exact(hip, oracle, shape, kv):
    w = weights(shape)
    g = hip.HipForward(shape, w, kv_capacity=512, max_chunk_rows=64, kv=kv)
    r = oracle.RefModel(shape, w, kv_bf16=(kv == "bf16"))
    prompt = synth.make_tokens(shape.vocab_size, 40, seed=3)
    ref_tokens = []
    logits = r.forward(prompt, 0, chunk_rows=16)
    for step in range(32):
        t = int(len(logits) - 1 - np.argmax(logits[::-1]))
        ref_tokens.append(t)
        logits = r.forward([t], 40 + step)
    first, = [g.forward_greedy(prompt, 0, chunk_rows=16)]
    assert first == ref_tokens[0]
    rest = g.decode_greedy(first, 40, 31)
    assert [first] + rest.tolist() == ref_tokens


@pytest.mark.parametrize("quant", [None, "q4"])
@pytest.mark.parametrize("shape", TINY, ids=lambda s: s.name)
def test_mixed_forward_calls_agree_with_device_greedy(hip, shape, quant):
    """forward (no sampling), forward_greedy with and without logits and
    decode_greedy in turn on one cache: the same tokens as decode_greedy alone
    and the same logit bits from either forward, on the persistent kernel and
    the decode graphs; the logits reach the host whole (an odd vocabulary ends
    inside a vector store)."""
    from cheetah_amd.workloads import greedy_token

    g = hip.HipForward(shape, weights(shape), quant=quant, kv_capacity=256, max_chunk_rows=32)
    prompt = synth.make_tokens(shape.vocab_size, 20, seed=4)
    first, logits = g.forward_greedy(prompt, 0, want_logits=True)
    assert first == greedy_token(logits)
    want = [first] + g.decode_greedy(first, 20, 8).tolist()
    g.clear_cache()
    assert np.array_equal(bits(g.forward(prompt, 0)), bits(logits))
    got = [first]
    got.append(greedy_token(g.forward(np.array(got[-1:], np.uint32), 20)))
    got.append(g.forward_greedy(np.array(got[-1:], np.uint32), 21))
    got += g.decode_greedy(got[-1], 22, 2).tolist()
    tok, lg = g.forward_greedy(np.array(got[-1:], np.uint32), 24, want_logits=True)
    assert tok == greedy_token(lg)
    got.append(tok)
    got.append(greedy_token(g.forward(np.array(got[-1:], np.uint32), 25)))
    got += g.decode_greedy(got[-1], 26, 2).tolist()
    assert got == want


@pytest.mark.parametrize("quant", [None, "q4"])
@pytest.mark.parametrize("shape", TINY, ids=lambda s: s.name)
def test_decode_logits_are_the_same_bits_with_and_without_sampling(hip, shape, quant):
    """One decode position on one restored cache through forward (no argmax) and
    forward_greedy, on the persistent kernel and the decode graphs, another
    token between them: all logits bit for bit, and the last ones (an odd
    vocabulary ends inside a vector store) not the other token's."""
    from cheetah_amd.workloads import greedy_token

    g = hip.HipForward(shape, weights(shape), quant=quant, kv_capacity=256, max_chunk_rows=32)
    prompt = synth.make_tokens(shape.vocab_size, 20, seed=14)
    g.forward(prompt, 0)
    snap = g.kv_snapshot()

    def at20(call, token):
        g.clear_cache()
        g.restore_kv_prefix(snap, 20)
        return call(np.array([token], np.uint32), 20)

    plain = at20(g.forward, 17)
    other = at20(g.forward, 401)
    token, logits = at20(lambda t, p: g.forward_greedy(t, p, want_logits=True), 17)
    assert np.array_equal(bits(plain), bits(logits))
    assert token == greedy_token(logits)
    tail = shape.vocab_size % 4 or 4
    assert (bits(other[-tail:]) != bits(logits[-tail:])).all()
    token, again = at20(lambda t, p: g.forward_greedy(t, p, want_logits=True), 401)
    assert np.array_equal(bits(other), bits(again)) and token == greedy_token(again)
    assert np.array_equal(bits(at20(g.forward, 17)), bits(logits))


def _attention64(q, k, v, group, offset):
    """q [rows, heads, hd] from position offset on, k/v [ctx, kv_heads, hd]; float64."""
    out = np.empty_like(q)
    for r in range(q.shape[0]):
        n = offset + r + 1
        for h in range(q.shape[1]):
            s = k[:n, h // group] @ q[r, h] / np.sqrt(q.shape[2])
            w = np.exp(s - s.max())
            out[r, h] = w @ v[:n, h // group] / w.sum()
    return out


@pytest.mark.parametrize("capacity", [640, 16384])
@pytest.mark.parametrize("q_heads,kv_heads,head_dim", [(2, 2, 64), (4, 2, 64), (7, 1, 64), (8, 1, 64), (4, 1, 128),
                                                       (7, 1, 128)])
def test_f32_kv_prefill_attention_holds_every_bit(hip, q_heads, kv_heads, head_dim, capacity):
    """The f32 prefill attention alone: queries are rotated biases, K and V are
    read back from layer 0, o_proj and layer 1's v_proj are identities, so layer
    1's V is the RMSNorm of embedding + attention. Against 64 bits, as 2-norms:
    two GEMM input splits (2^-18 / sqrt(3) each, 3e-6 together) and f32 scores of
    up to 42 (2e-6 where numpy sums them in f32): 1e-5. The same with the last 8
    bits of q, K and V cut off (the third parts left out) is 1.4e-5 to 3.4e-5 off."""
    dim = q_heads * head_dim
    kvd = kv_heads * head_dim
    shape = configs.TINY_QWEN2.replace(name=f"probe-{q_heads}-{kv_heads}-{head_dim}", hidden_size=dim, q_heads=q_heads,
                                       kv_heads=kv_heads, head_dim=head_dim)
    w = {k: synth.bf16_to_f32(v).copy() for k, v in synth.make_weights(shape).items()}
    p0, p1 = "model.layers.0.", "model.layers.1."
    rng = np.random.default_rng(q_heads + head_dim)
    scale = 8.0 / (0.02 * np.sqrt(dim))  # scores of 8 on average
    w[p0 + "self_attn.q_proj.weight"][:] = 0
    w[p0 + "self_attn.q_proj.bias"][:] = rng.standard_normal(dim) * scale
    w[p0 + "self_attn.o_proj.weight"][:] = np.eye(dim)
    w[p0 + "mlp.down_proj.weight"][:] = 0
    w[p1 + "self_attn.v_proj.weight"][:] = np.eye(dim)[:kvd]
    w[p1 + "self_attn.v_proj.bias"][:] = 0
    units = {k: synth.f32_to_bf16(v) for k, v in w.items()}
    g = hip.HipForward(shape, units, kv="f32", kv_capacity=capacity, max_chunk_rows=160)
    n, rows = 530, 24
    toks = synth.make_tokens(shape.vocab_size, n, seed=3)
    g.forward(toks, 0, chunk_rows=147)
    k, v = (t.astype(np.float64) for t in g.kv_rows(0, 0, n))
    got = g.kv_rows(1, n - rows, rows)[1].reshape(rows, kvd)

    half = head_dim // 2
    freq = np.power(np.float32(shape.rope_theta), np.float32(-2) * np.arange(half, dtype=np.float32) / np.float32(head_dim))
    angle = np.arange(n - rows, n, dtype=np.float32)[:, None] * freq.astype(np.float32)[None, :]
    cos, sin = (f(angle).astype(np.float32).astype(np.float64)[:, None, :] for f in (np.cos, np.sin))
    bias = synth.bf16_to_f32(units[p0 + "self_attn.q_proj.bias"]).astype(np.float64).reshape(1, q_heads, head_dim)
    a, b = bias[..., :half], bias[..., half:]
    q = np.concatenate([a * cos - b * sin, b * cos + a * sin], axis=-1).astype(np.float32).astype(np.float64)
    embed = synth.bf16_to_f32(units["model.embed_tokens.weight"])[toks[-rows:]].astype(np.float64)

    def layer1_v(q, k, v):
        x = embed + _attention64(q, k, v, q_heads // kv_heads, n - rows).reshape(rows, dim)
        return (x / np.sqrt((x * x).mean(axis=1, keepdims=True) + shape.rms_eps))[:, :kvd]

    def cut(t):
        return (t.astype(np.float32).view(np.uint32) & np.uint32(0xFFFFFF00)).view(np.float32).astype(np.float64)

    ref = layer1_v(q, k, v)
    off = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    assert off < 1e-5
    without = np.linalg.norm(layer1_v(cut(q), cut(k), cut(v)) - ref) / np.linalg.norm(ref)
    assert without > 1.2e-5


@pytest.mark.parametrize("shape", TINY, ids=lambda s: s.name)
def test_f32_kv_prefill_attention_tile_and_span_edges(hip, oracle, shape):
    """f32-cache prefill attention at the edges of its 64-key tiles, 256-key
    spans (capacity below 4,096) and row blocks, with a ragged chunk split.
    The attention itself is exact to f32 rounding; what is left against the
    oracle is the GEMMs' hi/lo input split: 2^-17 per product, averaged over a
    dot product, through 2 layers of 4 GEMMs on the largest logit: 5e-5."""
    g = hip.HipForward(shape, weights(shape), kv="f32", kv_capacity=640, max_chunk_rows=160)
    r = oracle.RefModel(shape, weights(shape))
    toks = synth.make_tokens(shape.vocab_size, 521, seed=21)
    for n, chunk in ((2, 160), (63, 160), (65, 64), (255, 33), (257, 160), (521, 147)):
        g.clear_cache()
        r.clear_cache()
        got = g.forward(toks[:n], 0, chunk_rows=chunk)
        ref = r.forward(toks[:n], 0, chunk_rows=256)
        assert rel_err(got, ref) < 5e-5, (n, chunk)


@pytest.mark.parametrize("shape", TINY, ids=lambda s: s.name)
def test_f32_kv_long_cache_bits_independent_of_chunks(hip, shape):
    """An f32 cache of 16,384 positions attends in splits of 2,048 keys, folded
    from parts of 256 in registers (chunks of 160 rows, whose parts the scratch
    does not hold) or by the merge (few rows): every position's K and V of the
    second layer and the last logits are the same bits either way, at the edges
    of parts and splits."""
    toks = synth.make_tokens(shape.vocab_size, 4200, seed=31)
    g = hip.HipForward(shape, weights(shape), kv="f32", kv_capacity=16384, max_chunk_rows=160)
    cuts = (0, 200, 255, 259, 510, 515, 2040, 2047, 2052, 2300, 4090, 4097, 4099, 4104, 4200)
    want = g.forward(toks, 0, chunk_rows=160)
    k0, v0 = g.kv_rows(1, 0, len(toks))
    g.clear_cache()
    for a, b in zip(cuts, cuts[1:]):
        got = g.forward(toks[a:b], a, chunk_rows=160 if b - a > 100 else 7)
    k1, v1 = g.kv_rows(1, 0, len(toks))
    assert np.array_equal(bits(k0), bits(k1)) and np.array_equal(bits(v0), bits(v1))
    assert np.array_equal(bits(got), bits(want))
    assert np.isfinite(want).all() and np.abs(k0).max() > 0


def _marked_model(head_dim, edit):
    """A two-layer qwen2 shape whose token 7 alone has a value at hidden unit 5
    (so a weight column 5 speaks of it alone), its units changed by
    `edit(units, shape)`: BF16 arrays by unit id."""
    shape = configs.TINY_QWEN2.replace(name=f"marked-{head_dim}", head_dim=head_dim)
    w = {k: synth.bf16_to_f32(v).copy() for k, v in synth.make_weights(shape).items()}
    w["model.embed_tokens.weight"][:, 5] = 0.0
    w["model.embed_tokens.weight"][7, 5] = 1.0
    edit(w, shape)
    return shape, {k: synth.f32_to_bf16(v) for k, v in w.items()}


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("capacity", [640, 16384])
def test_f32_kv_infinite_value_reaches_no_earlier_row(hip, head_dim, capacity):
    """Layer 0 gives token 7 infinite V values: the rows before it, in the same
    tile of the same call, keep the bits that a call without it gives them;
    the rows after it see the infinities."""
    def edit(w, shape):
        w["model.layers.0.self_attn.v_proj.weight"][3::64, 5] = 3e38

    shape, w = _marked_model(head_dim, edit)
    g = hip.HipForward(shape, w, kv="f32", kv_capacity=capacity, max_chunk_rows=160)
    toks = synth.make_tokens(shape.vocab_size, 300, seed=12)
    toks[toks == 7] = 8
    for at in (3, 70, 290):
        g.clear_cache()
        g.forward(toks[:at], 0, chunk_rows=160)
        want = g.kv_rows(1, 0, at)
        g.clear_cache()
        both = toks.copy()
        both[at] = 7
        assert not np.isfinite(g.forward(both, 0, chunk_rows=160)).all()
        assert np.isinf(g.kv_rows(0, at, 1)[1]).any()
        got = g.kv_rows(1, 0, at)
        for x, y in zip(got, want):
            assert np.isfinite(y).all()
            assert np.array_equal(bits(x), bits(y)), at


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("capacity", [640, 16384])
def test_f32_kv_nan_key_reaches_every_later_row_and_no_earlier_one(hip, head_dim, capacity):
    """Layer 0 gives token 7 NaN keys (an infinity through the rotation): every
    row from it on is NaN, whatever split the key is in, and the rows before it
    keep their bits."""
    def edit(w, shape):
        w["model.layers.0.self_attn.k_proj.weight"][:, 5] = 3e38 * np.where(np.arange(shape.kv_dim) % 2, 1, -1)

    shape, w = _marked_model(head_dim, edit)
    g = hip.HipForward(shape, w, kv="f32", kv_capacity=capacity, max_chunk_rows=160)
    toks = synth.make_tokens(shape.vocab_size, 600, seed=15)
    toks[toks == 7] = 8
    g.forward(toks, 0, chunk_rows=160)
    want = g.kv_rows(1, 0, 600)
    for at in (5, 300):
        g.clear_cache()
        both = toks.copy()
        both[at] = 7
        assert np.isnan(g.forward(both, 0, chunk_rows=160)).all()
        assert np.isnan(g.kv_rows(0, at, 1)[0]).any()
        for x, y in zip(g.kv_rows(1, 0, 600), want):
            assert np.array_equal(bits(x[:at]), bits(y[:at]))
            assert np.isnan(x[at:]).all()


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("capacity", [640, 16384])
def test_f32_kv_score_of_minus_infinity_weighs_nothing(hip, oracle, head_dim, capacity):
    """Token 7's keys and every query hold large values of opposite signs in the
    slowest rotary pair: their product is past the largest f32, -inf, and
    weighs nothing. The logits are finite and the oracle's within 5e-5 (the
    GEMMs' hi/lo input split, as in the tile and span edges test)."""
    def edit(w, shape):
        hd = shape.head_dim
        p = "model.layers.0.self_attn."
        w[p + "k_proj.weight"][hd // 2 - 1::hd, 5] = 1e29
        w[p + "q_proj.weight"][hd // 2 - 1::hd] = 0.0
        w[p + "q_proj.weight"][hd // 2 - 1::hd, 6:] = 1e13 * np.sign(w[p + "q_proj.weight"][:1, 6:] + 1e-6)
        w[p + "q_proj.bias"][hd // 2 - 1::hd] = -1e15

    shape, w = _marked_model(head_dim, edit)
    g = hip.HipForward(shape, w, kv="f32", kv_capacity=capacity, max_chunk_rows=160)
    r = oracle.RefModel(shape, w)
    toks = synth.make_tokens(shape.vocab_size, 300, seed=13)
    toks[toks == 7] = 8
    toks[[1, 40, 280]] = 7
    for n in (4, 60, 300):
        g.clear_cache()
        r.clear_cache()
        got = g.forward(toks[:n], 0, chunk_rows=160)
        ref = r.forward(toks[:n], 0, chunk_rows=256)
        assert np.isfinite(ref).all()
        assert rel_err(got, ref) < 5e-5, n


@pytest.mark.parametrize("kv", ["bf16", "f32"])
def test_kv_continuation_bit_exact_on_device(hip, kv):
    # decoder.rs:1710-1728: prefill in one call == prefill in two calls.
    shape = configs.TINY_QWEN2
    g = hip.HipForward(shape, weights(shape), kv_capacity=512, max_chunk_rows=64, kv=kv)
    toks = synth.make_tokens(shape.vocab_size, 90, seed=4)
    full = g.forward(toks[:70], 0, chunk_rows=32)
    dec_full = [g.forward(toks[i:i + 1], i) for i in range(70, 90)]
    g.clear_cache()
    g.forward(toks[:23], 0, chunk_rows=32)
    cont = g.forward(toks[23:70], 23, chunk_rows=16)
    assert np.array_equal(bits(full), bits(cont))
    for i in range(70, 90):
        assert np.array_equal(bits(g.forward(toks[i:i + 1], i)), bits(dec_full[i - 70])), i


def test_chunk_buffers_hold_what_a_chunk_reads(hip):
    """Device memory of 8,192 more chunk rows: the hidden, qkv and rotated query
    rows, the BF16 halves and the attention partials, and no f32 copies of the
    GEMMs' inputs (1 KiB + 32 KiB a row here). 100 MiB for split sums."""
    import ctypes

    runtime = ctypes.CDLL("libamdhip64.so.7")  # the one that the library runs on

    def free_bytes():
        free, total = ctypes.c_size_t(0), ctypes.c_size_t(0)
        assert runtime.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    shape = configs.TINY_QWEN2.replace(name="wide", intermediate_size=8192)
    units = synth.make_weights(shape)

    def used(rows):
        before = free_bytes()
        g = hip.HipForward(shape, units, kv_capacity=512, max_chunk_rows=rows)
        taken = before - free_bytes()
        g.close()
        return taken

    used(64)  # the library's first model: code and queues
    more = used(9216) - used(1024)
    inter, hidden, qd, kvd = shape.intermediate_size, shape.hidden_size, shape.q_dim, shape.kv_dim
    row = 4 * (hidden + 2 * qd + 2 * kvd) + 2 * 4 * inter + 4 * shape.q_heads * (shape.head_dim + 2)
    assert 8192 * row <= more < 8192 * row + (100 << 20), more / 8192


def test_snapshot_restore_clone_bit_exact_on_device(hip):
    # decoder.rs:1761-1818: a clone starts empty; snapshot -> restore ->
    # continue equals the uninterrupted run, including a restore that ends
    # mid-page (copy on write of the shared page).
    shape = configs.TINY_LLAMA
    g = hip.HipForward(shape, weights(shape), kv_capacity=1024, max_chunk_rows=64)
    toks = synth.make_tokens(shape.vocab_size, 150, seed=5)
    g.forward(toks[:130], 0, chunk_rows=64)
    snap = g.kv_snapshot()
    assert snap.positions == 130
    ref_next = [g.forward(toks[i:i + 1], i) for i in range(130, 150)]
    c = g.clone()
    assert c.kv_len() == 0
    for keep in (130, 100, 64):
        c.clear_cache()
        assert c.restore_kv_prefix(snap, keep)
        assert c.kv_len() == keep
        if keep < 130:
            c.forward(toks[keep:130], keep, chunk_rows=64)
        got = [c.forward(toks[i:i + 1], i) for i in range(130, 150)]
        for a, b in zip(got, ref_next):
            if keep == 130:
                assert np.array_equal(bits(a), bits(b))
            else:
                assert rel_err(a, b) < 1e-4  # re-prefilled tail: same math, prefill kernels
    # the original keeps its own cache untouched by the clone's writes
    g.clear_cache()
    g.forward(toks[:130], 0, chunk_rows=64)
    again = g.forward(toks[130:131], 130)
    assert np.array_equal(bits(again), bits(ref_next[0]))


def test_restore_then_continue_matches_full_prefill_bit_exact(hip):
    # The engine's prefix reuse (engine.rs:1880-1890): restoring n cached
    # positions then prefilling the suffix gives the same logits as the
    # uninterrupted prefill, bit for bit (prefill split boundaries depend only
    # on each row's position).
    shape = configs.TINY_QWEN2
    g = hip.HipForward(shape, weights(shape), kv_capacity=1024, max_chunk_rows=64)
    toks = synth.make_tokens(shape.vocab_size, 200, seed=6)
    full = g.forward(toks, 0, chunk_rows=64)
    snap = g.kv_snapshot()
    c = g.clone()
    c.restore_kv_prefix(snap, 150)
    cont = c.forward(toks[150:], 150, chunk_rows=64)
    assert np.array_equal(bits(full), bits(cont))


def test_forward_errors_are_reported_before_device_work(hip):
    shape = configs.TINY_QWEN2
    g = hip.HipForward(shape, weights(shape), kv_capacity=128, max_chunk_rows=64)
    with pytest.raises(hip.HipError, match="empty token input"):
        g.forward(np.array([], np.uint32), 0)
    with pytest.raises(hip.HipError, match="exceeds the vocabulary size 1000"):
        g.forward(np.array([5, 1000], np.uint32), 0)
    with pytest.raises(hip.HipError, match="does not match the input offset"):
        g.forward(np.array([5], np.uint32), 3)
    with pytest.raises(hip.HipError, match="capacity"):
        g.forward(np.zeros(129, np.uint32), 0)
    assert g.kv_len() == 0
    g.forward(np.array([5, 6], np.uint32), 0)
    assert g.kv_len() == 2


def test_missing_unit_is_rejected(hip):
    shape = configs.TINY_QWEN2
    w = dict(weights(shape))
    del w["model.layers.1.mlp.down_proj.weight"]
    with pytest.raises(hip.HipError, match="missing unit 'model.layers.1.mlp.down_proj.weight'"):
        hip.HipForward(shape, w)


def test_pool_exhaustion_mid_reserve_leaves_shared_pages_intact(hip):
    """A forward that runs out of KV pages part way through mapping its
    positions fails and changes nothing: the page it copied on write goes
    back to the pool and the instance keeps mapping the shared page, so a
    retry copies again instead of writing through a stale device table into
    the page a snapshot holds."""
    shape = configs.TINY_QWEN2
    toks = synth.make_tokens(shape.vocab_size, 200, seed=12)
    other = synth.make_tokens(shape.vocab_size, 10, seed=13)

    def run(prefix, tail, at):
        r = hip.HipForward(shape, weights(shape), kv_capacity=512, max_chunk_rows=64)
        r.forward(prefix, 0, chunk_rows=64)
        out = r.forward(tail, at, chunk_rows=64)
        r.close()
        return out

    want_retry = run(toks[:130], other, 130)
    want_snap = run(toks[:150], toks[150:160], 150)
    # 256 positions = 4 pages. The snapshot holds positions 0..149 (pages
    # 0-2); the model maps the first 130 of them, sharing all three pages.
    g = hip.HipForward(shape, weights(shape), kv_capacity=256, max_chunk_rows=64)
    g.forward(toks[:150], 0, chunk_rows=64)
    snap = g.kv_snapshot()
    g.clear_cache()
    assert g.restore_kv_prefix(snap, 130)
    # Positions 130..199 need a copy of page 2 (the one free page) and a new
    # page 3 (none left): the call fails after the copy.
    with pytest.raises(hip.HipError, match="KV page pool exhausted"):
        g.forward(toks[130:200], 130, chunk_rows=64)
    assert g.kv_len() == 130
    # The retry writes positions 130..139 of page 2, which the snapshot
    # holds with other values.
    got = g.forward(other, 130, chunk_rows=64)
    assert np.array_equal(bits(got), bits(want_retry))
    g.clear_cache()
    c = g.clone()
    assert c.restore_kv_prefix(snap, 150)
    again = c.forward(toks[150:160], 150, chunk_rows=64)
    assert np.array_equal(bits(again), bits(want_snap))
    c.close()
    g.close()


def _qwen2_greedy(hip, kv, gold):
    """Prefill, then greedy decode: the device greedy loop, with the logits of
    decode steps 1, 16 and 32 taken through the per-step forward."""
    shape = configs.QWEN2_0_5B
    g = hip.HipForward(shape, weights(shape), kv_capacity=1024, max_chunk_rows=128, kv=kv)
    prompt = synth.make_tokens(shape.vocab_size, gold["prompt_len"], seed=gold["prompt_seed"])
    first, logits = g.forward_greedy(prompt, 0, chunk_rows=gold["chunk_rows"], want_logits=True)
    tokens, dec_logits = golden_checks.decode_sampled(g, first, gold["prompt_len"], len(gold["tokens"]))
    g.close()
    return logits, tokens, dec_logits


def _gold(name):
    with open(os.path.join(GOLDEN, name)) as f:
        return json.load(f)


def test_qwen2_0_5b_greedy_f32_kv_matches_reference(hip):
    """Config 1 (Qwen2-0.5B shape, BF16 weights): 512-token prompt prefilled
    in chunks of 128, then greedy decode. With the reference's own f32 KV
    cache the first 32 tokens equal the CPU path's (golden from
    tests/golden/make_golden.py)."""
    gold = _gold("qwen2_0_5b_greedy.json")
    logits, got, dec = _qwen2_greedy(hip, "f32", gold)
    head = np.array(gold["prefill_logits_head"], np.float32)
    assert rel_err(logits[: head.size], head) < 1e-2
    golden_checks.check_vocab_sample(logits, gold["prefill_vocab_sample"], what="prefill")
    assert got[:32] == gold["tokens"][:32], got
    errs = golden_checks.check_decode_samples(dec, got, gold)
    assert sorted(errs) == [1, 16, 32], errs


def test_qwen2_0_5b_greedy_bf16_kv(hip):
    """The BF16 paged KV cache (the served default) equals the oracle run
    with BF16-rounded K/V for 64 steps; against the f32-KV reference it
    departs only at a near-tie: at the first differing step the reference's
    top-2 margin is below 0.01 (0.0042 at step 23 for this seed)."""
    gold_bf = _gold("qwen2_0_5b_bf16kv_greedy.json")
    gold_ref = _gold("qwen2_0_5b_greedy.json")
    logits, got, dec = _qwen2_greedy(hip, "bf16", gold_bf)
    head = np.array(gold_ref["prefill_logits_head"], np.float32)
    assert rel_err(logits[: head.size], head) < 1e-2
    golden_checks.check_vocab_sample(logits, gold_bf["prefill_vocab_sample"], what="prefill")
    golden_checks.check_vocab_sample(logits, gold_ref["prefill_vocab_sample"], what="prefill vs f32-KV reference")
    assert got == gold_bf["tokens"], got
    errs = golden_checks.check_decode_samples(dec, got, gold_bf)
    assert sorted(errs) == [1, 16, 32], errs
    golden_checks.check_departure_at_near_tie(got, gold_ref, n=len(got), margin_bar=1e-2)


@pytest.mark.parametrize("kv", ["bf16", "f32"])
@pytest.mark.parametrize("shape", TINY + [configs.QWEN2_0_5B], ids=lambda s: s.name)
def test_persistent_decode_matches_graph_decode(hip, shape, kv, monkeypatch):
    """The persistent decode kernel (one launch for many steps, no
    device-wide barrier) and the per-step graph path compute the same math:
    same greedy tokens over 40 steps and logits within 1e-4 relative."""
    w = weights(shape)
    prompt = synth.make_tokens(shape.vocab_size, 100, seed=11)
    runs = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("CHEETAH_HIP_FUSED", mode)
        g = hip.HipForward(shape, w, kv_capacity=1024, max_chunk_rows=64, kv=kv)
        first = g.forward_greedy(prompt, 0, chunk_rows=64)
        toks = g.decode_greedy(first, 100, 40)
        logits = g.forward(toks[-1:], 140)
        runs[mode] = ([first] + toks.tolist(), logits)
        g.close()
    assert runs["1"][0] == runs["0"][0]
    assert rel_err(runs["1"][1], runs["0"][1]) < 1e-4


def test_persistent_decode_long_runs_match_graph_decode(hip, monkeypatch):
    """Near the persistent kernel's longest context (Qwen2-0.5B, BF16 K/V: 5
    runs of 256 positions, 1,280), a 900-token prompt and 40 steps take
    256-position attention runs: each wave of an item scores up to 32 cached
    positions in four passes of 8, a run's last wave a partial pass. Same
    greedy tokens as the graph path and logits within 1e-4."""
    shape = configs.QWEN2_0_5B
    w = weights(shape)
    prompt = synth.make_tokens(shape.vocab_size, 900, seed=17)
    runs = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("CHEETAH_HIP_FUSED", mode)
        g = hip.HipForward(shape, w, kv_capacity=1024, max_chunk_rows=128, kv="bf16")
        first = g.forward_greedy(prompt, 0, chunk_rows=128)
        toks = g.decode_greedy(first, 900, 40)
        logits = g.forward(toks[-1:], 940)
        runs[mode] = ([first] + toks.tolist(), logits)
        g.close()
    assert runs["1"][0] == runs["0"][0]
    assert rel_err(runs["1"][1], runs["0"][1]) < 1e-4


@pytest.mark.parametrize("shape,quant,big", [(configs.QWEN2_0_5B, None, 2048),
                                              (configs.LLAMA3_8B.replace(num_layers=2), "q4", 512)],
                         ids=["qwen2-0.5b-bf16", "llama3-8b-2layer-q4"])
def test_prefill_bits_independent_of_split_k(hip, shape, quant, big):
    """A big chunk gives the QKV and gate/up GEMMs enough tiles to fold K in
    registers (gate/up on 128-token tiles); 128-row chunks split K and fold
    the chunk sums in the RoPE kernel and the SwiGLU reduce. Both follow the
    same chunk order, so the last row's logits are the same bits
    (decoder.rs:1710-1728: a position's result does not depend on how the
    prompt was cut)."""
    g = hip.HipForward(shape, weights(shape), quant=quant, kv_capacity=big + 64, max_chunk_rows=big)
    try:
        toks = synth.make_tokens(shape.vocab_size, big, seed=6)
        whole = g.forward(toks, 0, chunk_rows=big)
        g.clear_cache()
        chunked = g.forward(toks, 0, chunk_rows=128)
        assert np.array_equal(bits(whole), bits(chunked))
    finally:
        g.close()
