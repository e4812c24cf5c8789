"""Op-level parity of the HIP kernels against the CPU oracle, through the C-ABI.

Bars (north star): Q8/Q4 dequantized values bit-exact; GEMV / GEMM /
attention outputs within 1e-2 relative (f32 accumulation). The asserts
below are tighter where both sides accumulate in f32.
"""
import numpy as np
import pytest

from cheetah_amd import synth

pytestmark = pytest.mark.gpu

REL_BAR = 1e-2  # north-star tolerance for floating-point outputs


@pytest.fixture(scope="module")
def hip():
    from cheetah_amd import hip as h
    h.init(0)
    return h


def rel_err(got, ref):
    got = np.asarray(got, np.float64)
    ref = np.asarray(ref, np.float64)
    return float(np.max(np.abs(got - ref)) / max(np.max(np.abs(ref)), 1e-30))


def random_quant(rng, fmt, rows, cols):
    """Config-3 style buffer: codes uniform over the full range, scales U[1e-3, 1e-2]."""
    scales = rng.uniform(1e-3, 1e-2, rows).astype(np.float32)
    if fmt == "q8":
        stride = (cols + 3) // 4 * 4
        codes = rng.integers(-127, 128, (rows, cols)).astype(np.int8)
        payload = np.zeros((rows, stride), np.uint8)
        payload[:, :cols] = codes.view(np.uint8)
    else:
        stride = ((cols + 2) // 2 + 3) // 4 * 4
        codes = rng.integers(-8, 8, (rows, cols)).astype(np.int16)
        payload = np.zeros((rows, stride), np.uint8)
        nib = (codes & 0xF).astype(np.uint8)
        payload[:, : (cols + 1) // 2] |= nib[:, 0::2]
        payload[:, : cols // 2] |= (nib[:, 1::2] << 4)
    return np.concatenate([scales.view(np.uint8), payload.reshape(-1)])


GEMV_SHAPES = [(1, 1), (3, 9), (5, 17), (64, 100), (130, 896), (259, 1000), (896, 4864), (1152, 896)]


@pytest.mark.parametrize("fmt", ["bf16", "q8", "q4"])
@pytest.mark.parametrize("rows,cols", GEMV_SHAPES)
def test_gemv_matches_oracle(hip, oracle, fmt, rows, cols):
    rng = np.random.default_rng(rows * 1000 + cols)
    x = rng.standard_normal(cols).astype(np.float32)
    if fmt == "bf16":
        w = synth.f32_to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
        ref = oracle.gemv(w, x)
        wd = hip.DeviceBuffer.from_array(w)
    else:
        buf = random_quant(rng, fmt, rows, cols)
        ref = oracle.gemv_quant(buf, rows, cols, x, fmt)
        wd = hip.DeviceBuffer.from_array(buf)
    got = hip.gemv(wd, fmt, rows, cols, x)
    assert rel_err(got, ref) < 1e-5 < REL_BAR


@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("rows,cols", [(3, 9), (4096, 4096), (4096, 14336), (14336, 4096)])
def test_config3_gemv_shapes(hip, oracle, fmt, rows, cols):
    rng = np.random.default_rng(7)
    buf = random_quant(rng, fmt, rows, cols)
    x = synth.bf16_to_f32(synth.f32_to_bf16(rng.standard_normal(cols).astype(np.float32)))
    ref = oracle.gemv_quant(buf, rows, cols, x, fmt)
    got = hip.gemv(hip.DeviceBuffer.from_array(buf), fmt, rows, cols, x)
    assert rel_err(got, ref) < 1e-5


@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("rows,cols", [(3, 9), (8, 64), (37, 1001), (256, 4096)])
def test_quantize_and_dequant_bit_exact(hip, oracle, fmt, rows, cols):
    rng = np.random.default_rng(rows + cols)
    w = synth.f32_to_bf16((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    w[0, :] = 0  # zero row: scale 1.0
    if rows > 2:  # exact ties: max|w| = 7 * 2^k makes w/scale hit .5 exactly
        w[1, :4] = synth.f32_to_bf16(np.array([7.0, 2.5, -2.5, 0.5], np.float32))
    values = synth.bf16_to_f32(w).reshape(rows, cols)
    ref = oracle.quantize(values, fmt)
    got = hip.quantize(w, fmt)
    assert np.array_equal(got, ref)
    deq = hip.dequant(got, fmt, rows, cols)
    assert np.array_equal(deq.view(np.uint32), oracle.dequant(ref, rows, cols, fmt).view(np.uint32))


@pytest.mark.parametrize("fmt", ["bf16", "q8", "q4"])
@pytest.mark.parametrize("n,rows,cols", [(1, 5, 9), (7, 259, 100), (64, 128, 896), (130, 300, 1000),
                                         (128, 1152, 896)])
def test_gemm_matches_oracle(hip, oracle, fmt, n, rows, cols):
    rng = np.random.default_rng(n * 7 + rows)
    x = rng.standard_normal((n, cols)).astype(np.float32)
    if fmt == "bf16":
        w = synth.f32_to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
        ref = oracle.gemm_bf16(w, x)
        wd = hip.DeviceBuffer.from_array(w)
    else:
        buf = random_quant(rng, fmt, rows, cols)
        ref = np.stack([oracle.gemv_quant(buf, rows, cols, x[t], fmt) for t in range(n)])
        wd = hip.DeviceBuffer.from_array(buf)
    got = hip.gemm(wd, fmt, rows, cols, x)
    assert rel_err(got, ref) < 1e-4 < REL_BAR


@pytest.mark.parametrize("fmt", ["bf16", "q4"])
def test_config3_gemm_prefill_chunk(hip, oracle, fmt):
    # N = 512 against 4096 x 4096 (the prefill-chunk case of the GEMV/GEMM op).
    rng = np.random.default_rng(11)
    rows = cols = 4096
    n = 512
    x = synth.bf16_to_f32(synth.f32_to_bf16(rng.standard_normal((n, cols)).astype(np.float32))).reshape(n, cols)
    if fmt == "bf16":
        w = synth.f32_to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
        ref = oracle.gemm_bf16(w, x)
        wd = hip.DeviceBuffer.from_array(w)
    else:
        buf = random_quant(rng, fmt, rows, cols)
        sel = np.arange(0, n, 37)
        ref = np.stack([oracle.gemv_quant(buf, rows, cols, x[t], fmt) for t in sel])
        wd = hip.DeviceBuffer.from_array(buf)
    got = hip.gemm(wd, fmt, rows, cols, x)
    if fmt != "bf16":
        got = got[sel]
    assert rel_err(got, ref) < 1e-4


@pytest.mark.parametrize("fmt", ["bf16", "q8", "q4"])
def test_gemm_bits_independent_of_token_count(hip, fmt):
    """4096 x 4096 weights (16 accumulation chunks of 256) on 256 CUs: 1,024
    tokens fold K in registers on 8-wave blocks, 512 tokens run the two chunk
    halves as separate 8-wave blocks (half sums folded by the reduce), 128
    tokens one block per chunk (all 16 sums folded by the reduce). Each path
    folds the chunks as two halves, so a token's outputs are the same bits in
    all three (a prompt's results do not depend on how it is chunked)."""
    rng = np.random.default_rng(5)
    rows = cols = 4096
    x = rng.standard_normal((1024, cols)).astype(np.float32)
    if fmt == "bf16":
        wd = hip.DeviceBuffer.from_array(synth.f32_to_bf16(rng.standard_normal((rows, cols)).astype(np.float32)))
    else:
        wd = hip.DeviceBuffer.from_array(random_quant(rng, fmt, rows, cols))

    def bits(a):
        return np.ascontiguousarray(a, np.float32).view(np.uint32)

    y1024 = hip.gemm(wd, fmt, rows, cols, x)
    y512 = hip.gemm(wd, fmt, rows, cols, x[:512])
    y128 = hip.gemm(wd, fmt, rows, cols, x[:128])
    assert np.array_equal(bits(y1024[:512]), bits(y512))
    assert np.array_equal(bits(y512[:128]), bits(y128))
    assert np.isfinite(y1024).all() and np.abs(y1024).max() > 0


@pytest.mark.parametrize("fmt", ["bf16", "q8", "q4"])
@pytest.mark.parametrize("rows,cols", [(1001, 64), (515, 896), (4097, 4096), (14336, 1024), (130, 33), (259, 1001),
                                       (4096, 1009), (9001, 2048)])
def test_gemm_tile_edges_give_the_same_bits(hip, oracle, fmt, rows, cols):
    """Token counts and row counts around the edges of the 64 / 128-token and
    128 / 256-row tiles, odd row counts (Q8 payloads only 4-byte aligned) and
    every K split the sizes choose (9001 x 2048 at 1,030 tokens: full rounds
    of large tiles, then the rest on smaller ones), with column counts that end inside a
    32-column stage (Q8/Q4 on zero-padded input halves): a token's outputs are the same bits in
    every call, and the oracle's within the hi/lo input split (2^-17 per
    product; 1e-5 of the largest output)."""
    rng = np.random.default_rng(rows + cols)
    x = rng.standard_normal((1030, cols)).astype(np.float32)
    if fmt == "bf16":
        w = synth.f32_to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
        wd = hip.DeviceBuffer.from_array(w)
    else:
        buf = random_quant(rng, fmt, rows, cols)
        wd = hip.DeviceBuffer.from_array(buf)
    full = np.ascontiguousarray(hip.gemm(wd, fmt, rows, cols, x))
    for n in (1, 63, 64, 65, 128, 129, 257, 389, 512):
        got = np.ascontiguousarray(hip.gemm(wd, fmt, rows, cols, x[:n]))
        assert np.array_equal(got.view(np.uint32), full[:n].view(np.uint32)), n
    sel = np.array([0, 63, 64, 127, 128, 1023, 1024, 1029])
    xs = np.ascontiguousarray(x[sel])
    ref = oracle.gemm_bf16(w, xs) if fmt == "bf16" else oracle.gemm_quant(buf, rows, cols, xs, fmt)
    assert rel_err(full[sel], ref) < 1e-5


@pytest.mark.parametrize("fmt", ["bf16", "q8", "q4"])
@pytest.mark.parametrize("rows,cols", [(2240, 128), (640, 160), (20000, 2048), (4096, 2304)])
def test_gemm_few_tokens_and_few_columns_give_the_same_bits(hip, oracle, fmt, rows, cols):
    """Few columns (unsplit or per chunk by the token count) and the weight
    stream of few tokens: BF16 on the five-stage ring (20000 x 2048, over four
    blocks a CU) and on the four-stage one (4096 x 2304, one to four): the same
    bits at every token count, and the oracle's within the hi/lo input split
    (2^-17 per product; 1e-5 of the largest output)."""
    rng = np.random.default_rng(rows + 3 * cols)
    x = rng.standard_normal((130, cols)).astype(np.float32)
    if fmt == "bf16":
        w = synth.f32_to_bf16(rng.standard_normal((rows, cols)).astype(np.float32))
        wd = hip.DeviceBuffer.from_array(w)
    else:
        buf = random_quant(rng, fmt, rows, cols)
        wd = hip.DeviceBuffer.from_array(buf)
    full = np.ascontiguousarray(hip.gemm(wd, fmt, rows, cols, x))
    for n in (1, 8, 9, 37, 64, 65):
        got = np.ascontiguousarray(hip.gemm(wd, fmt, rows, cols, x[:n]))
        assert np.array_equal(got.view(np.uint32), full[:n].view(np.uint32)), n
    sel = np.array([0, 36, 64, 129])
    xs = np.ascontiguousarray(x[sel])
    ref = oracle.gemm_bf16(w, xs) if fmt == "bf16" else oracle.gemm_quant(buf, rows, cols, xs, fmt)
    assert rel_err(full[sel], ref) < 1e-5


def _attn_case(rng, q_heads, kv_heads, hd, ctx, rows):
    k = synth.f32_to_bf16(rng.standard_normal((ctx, kv_heads, hd)).astype(np.float32))
    v = synth.f32_to_bf16(rng.standard_normal((ctx, kv_heads, hd)).astype(np.float32))
    q = rng.standard_normal((rows, q_heads * hd)).astype(np.float32)
    return k, v, q


@pytest.mark.parametrize("fmt", ["bf16", "q8", "q4"])
@pytest.mark.parametrize("cols", [32, 33, 40])
def test_gemm_refuses_an_input_off_16_bytes(hip, fmt, cols):
    """Every format and column count, padded to whole stages or not."""
    rng = np.random.default_rng(cols)
    rows, n = 8, 3
    w = rng.integers(0, 16000, (rows, cols)).astype(np.uint16) if fmt == "bf16" else random_quant(rng, fmt, rows, cols)
    wd = hip.DeviceBuffer.from_array(w)
    xd = hip.DeviceBuffer.from_array(np.zeros(n * cols + 4, np.float32))
    yd = hip.DeviceBuffer(n * rows * 4)
    fn = getattr(hip.lib(), f"cheetah_hip_gemm_{fmt}")
    for off in (4, 8, 12):
        with pytest.raises(hip.HipError, match="aligned"):
            hip.check(fn(wd.ptr, rows, cols, xd.ptr + off, n, yd.ptr))
    hip.check(fn(wd.ptr, rows, cols, xd.ptr + 16, n, yd.ptr))


@pytest.mark.parametrize("rows,cols", [(0, 64), (64, 0)])
def test_time_gemm_refuses_an_empty_matrix(hip, rows, cols):
    """Before its workspace is planned (a division by the column count)."""
    import ctypes

    buf = hip.DeviceBuffer(4096)
    ms = ctypes.c_float(0)
    with pytest.raises(hip.HipError, match="columns"):
        hip.check(hip.lib().cheetah_hip_time_gemm(1, (ctypes.c_void_p * 1)(buf.ptr), 1, rows, cols, buf.ptr, 4, buf.ptr,
                                                  1, ctypes.byref(ms)))


@pytest.mark.parametrize("q_heads,kv_heads,hd", [(14, 2, 64), (32, 8, 128), (28, 4, 128), (4, 4, 64), (8, 1, 64)])
@pytest.mark.parametrize("ctx", [1, 63, 64, 65, 1000, 4096])
def test_attention_decode_matches_oracle(hip, oracle, q_heads, kv_heads, hd, ctx):
    rng = np.random.default_rng(ctx + q_heads)
    k, v, q = _attn_case(rng, q_heads, kv_heads, hd, ctx, 1)
    kp, vp, table = hip.paged_kv(k, v, seed=ctx)
    got = hip.attention(q, kp, vp, table, q_heads, 1, ctx - 1)[0]
    ref = oracle.attention(synth.bf16_to_f32(k), synth.bf16_to_f32(v), q[0], q_heads, kv_heads, hd, ctx - 1)
    assert np.max(np.abs(got - ref)) < 1e-4


@pytest.mark.parametrize("q_heads,kv_heads,hd,ctx", [(14, 2, 64, 128), (14, 2, 64, 129), (14, 2, 64, 384),
                                                     (14, 2, 64, 385), (32, 8, 128, 97), (28, 4, 128, 256),
                                                     (28, 4, 128, 257), (8, 1, 128, 255)])
def test_attention_decode_around_the_one_block_limit(hip, oracle, q_heads, kv_heads, hd, ctx):
    """Short contexts run as one block per KV head (256 keys at head_dim 128,
    384 at 64), longer ones split and merge: the edges of both, and of the
    rounds of four 32-key tiles. Queries and probabilities are two BF16 halves
    (2^-17); values are N(0, 1): 2e-5 of the output's scale."""
    rng = np.random.default_rng(ctx + hd)
    k, v, q = _attn_case(rng, q_heads, kv_heads, hd, ctx, 1)
    kp, vp, table = hip.paged_kv(k, v, seed=ctx)
    got = hip.attention(q, kp, vp, table, q_heads, 1, ctx - 1)[0]
    ref = oracle.attention(synth.bf16_to_f32(k), synth.bf16_to_f32(v), q[0], q_heads, kv_heads, hd, ctx - 1)
    assert rel_err(got, ref) < 2e-5


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("ctx", [65536, 65537, 131072])
def test_attention_prefill_merges_more_than_64_splits(hip, hd, ctx):
    """Two rows at the end of a long context: 64, 65 and 128 splits of 1,024
    keys, two a lane in the merge, against the same in 64 bits. Queries and
    probabilities are two BF16 halves (2^-17 per product, averaged over the keys
    as the output is): 2e-5 of the largest output."""
    rng = np.random.default_rng(ctx + hd)
    k, v, q = _attn_case(rng, 2, 1, hd, ctx, 2)
    kp, vp, table = hip.paged_kv(k, v, seed=7)
    got = hip.attention(q, kp, vp, table, 2, 2, ctx - 2).reshape(2, 2, hd)
    kf, vf = (synth.bf16_to_f32(t)[:, 0].astype(np.float64) for t in (k, v))
    for row in range(2):
        n = ctx - 1 + row
        s = q[row].reshape(2, hd).astype(np.float64) @ kf[:n].T / np.sqrt(hd)
        w = np.exp(s - s.max(axis=1, keepdims=True))
        ref = w @ vf[:n] / w.sum(axis=1, keepdims=True)
        assert rel_err(got[row], ref) < 2e-5, row


@pytest.mark.parametrize("q_heads,kv_heads,hd", [(14, 2, 64), (16, 2, 64), (3, 1, 64), (32, 8, 128), (10, 2, 128)])
@pytest.mark.parametrize("ctx,rows", [(37, 37), (63, 2), (64, 64), (65, 33), (127, 127), (129, 70), (1023, 65), (1025, 40),
                                      (2113, 9)])
def test_attention_prefill_tile_and_span_edges_with_unwritten_rows(hip, oracle, q_heads, kv_heads, hd, ctx, rows):
    """Prefill at the edges of the 64-key tiles and the 1,024-key spans, ragged
    row blocks, several tiles (rescaling, both buffers) and the split merge,
    with NaN in the rows of the last page past the context: cache memory that
    nothing has written yet, which a probability of 0 does not clear. Queries and
    probabilities are two BF16 halves (2^-17): 2e-5 of the largest output."""
    rng = np.random.default_rng(ctx + hd + q_heads)
    k, v, q = _attn_case(rng, q_heads, kv_heads, hd, ctx, rows)
    kp, vp, table = hip.paged_kv(k, v, seed=ctx)
    if ctx % 64:
        kp[table[-1], :, ctx % 64:] = 0x7FC0
        vp[table[-1], :, ctx % 64:] = 0x7FC0
    got = hip.attention(q, kp, vp, table, q_heads, rows, ctx - rows)
    ref = oracle.attention_rows(synth.bf16_to_f32(k), synth.bf16_to_f32(v), q, q_heads, kv_heads, hd, ctx - rows)
    assert np.isfinite(got).all()
    assert rel_err(got, ref) < 2e-5


def test_attention_prefill_first_calls_from_several_threads(hip, oracle):
    """The first call of a kernel lets it take its LDS, from whichever thread
    comes first: eight threads at once, each with its own buffers and scratch."""
    import threading

    rng = np.random.default_rng(11)
    k, v, q = _attn_case(rng, 15, 5, 128, 70, 6)
    kp, vp, table = hip.paged_kv(k, v, seed=2)
    got = [None] * 8

    def run(i):
        got[i] = hip.attention(q, kp, vp, table, 15, 6, 64)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    kf, vf = synth.bf16_to_f32(k), synth.bf16_to_f32(v)
    ref = oracle.attention_rows(kf, vf, q, 15, 5, 128, 64)
    for g in got:
        assert np.max(np.abs(g - ref)) < 1e-4


@pytest.mark.parametrize("q_heads,kv_heads,hd,offset,rows", [(14, 2, 64, 0, 37), (32, 8, 128, 100, 70),
                                                            (28, 4, 128, 4000, 9)])
def test_attention_prefill_rows_match_oracle(hip, oracle, q_heads, kv_heads, hd, offset, rows):
    rng = np.random.default_rng(offset + rows)
    ctx = offset + rows
    k, v, q = _attn_case(rng, q_heads, kv_heads, hd, ctx, rows)
    kp, vp, table = hip.paged_kv(k, v, seed=rows)
    got = hip.attention(q, kp, vp, table, q_heads, rows, offset)
    kf, vf = synth.bf16_to_f32(k), synth.bf16_to_f32(v)
    for i in range(rows):
        pos = offset + i
        ref = oracle.attention(kf[: pos + 1], vf[: pos + 1], q[i], q_heads, kv_heads, hd, pos)
        assert np.max(np.abs(got[i] - ref)) < 1e-4, i


def test_attention_two_token_gqa_kat(hip):
    # native.rs:2017-2033 closed form, through the paged kernel (hd padded to
    # 64 with zeros; zero dims change neither scores nor outputs... except the
    # 1/sqrt(head_dim) scale, so the expected weights use hd = 64).
    hd = 64
    k = np.zeros((2, 1, hd), np.float32)
    v = np.zeros((2, 1, hd), np.float32)
    k[0, 0, 0] = 1.0
    k[1, 0, 1] = 1.0
    v[0, 0, :2] = [2.0, 3.0]
    v[1, 0, :2] = [5.0, 7.0]
    q = np.zeros((1, 2 * hd), np.float32)
    q[0, 0] = 1.0
    q[0, hd + 1] = 1.0
    kp, vp, table = hip.paged_kv(synth.f32_to_bf16(k), synth.f32_to_bf16(v))
    out = hip.attention(q, kp, vp, table, 2, 1, 1)[0]
    w = 1.0 / (1.0 + np.exp(-1.0 / np.sqrt(hd)))
    exp0 = [2 * w + 5 * (1 - w), 3 * w + 7 * (1 - w)]
    exp1 = [2 * (1 - w) + 5 * w, 3 * (1 - w) + 7 * w]
    assert np.allclose(out[:2], exp0, atol=1e-5) and np.allclose(out[hd:hd + 2], exp1, atol=1e-5)
