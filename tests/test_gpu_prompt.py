"""The kernels of a prompt pass at the edges of their tiles: the matmul over 17 and more rows for every storage type, attention
over consecutive rows, and whole prompts at lengths around the passes' limits."""
import numpy as np
import pytest

from oracle import binding as ob
from tests import gpu_common as gc
from tests.test_oracle_quant import lcg_weights

pytestmark = pytest.mark.gpu


# rows and columns around the 128-column tiles and the 256-, 128- and 64-wide chunks; m around the 64-, 128- and 256-row tiles
@pytest.mark.parametrize("dtype,rows,cols", [(12, 64, 512), (12, 200, 768), (13, 64, 512), (13, 200, 768), (14, 130, 512), (14, 64, 1024),
                                             (8, 64, 128), (8, 200, 1408), (30, 64, 64), (30, 130, 2880), (39, 64, 256), (39, 200, 2880)])
@pytest.mark.parametrize("m", [17, 64, 65, 128, 129, 257, 321])
def test_the_prompt_matmul_is_the_dequantized_product(dtype, rows, cols, m):
    from turbospark_amd import ffi
    w = lcg_weights(rows * cols, 5).reshape(rows, cols) * 0.05
    w[::7] *= 1e-3                                     # rows and blocks of very different scale
    w[3, :cols // 2] *= 1e-2
    w[5, :32] = w[9] = 0.0                             # a zero block, a zero row
    entry = ffi.quantize(dtype, w)
    x = lcg_weights(m * cols, 6).reshape(m, cols)
    deq = ob.dequantize(dtype, entry[1], cols).astype(np.float64)
    want = x.astype(np.float16).astype(np.float64) @ deq.T
    # fp32 sums of exact products: rounding of about sqrt(K) terms of the row's size (the bound of the 16-row kernels' test)
    scale = np.abs(want).max(0)
    for splits in (0, 1):
        got = ffi.matmul(entry, x, splits)
        assert (np.abs(got - want) <= 2e-4 * scale + 1e-9).all(), (splits, np.abs(got - want).max() / scale.max())
        # and column by column: K / 16 sums in one chain, twice that for weights of two terms, each rounded to 2^-24 of the running
        # size; four times that covers the min terms of Q4_K / Q5_K, larger than what they leave
        norm = np.linalg.norm(want, axis=0)
        assert (np.linalg.norm(got - want, axis=0) <= 4 * (cols / 16) ** 0.5 * 2.0 ** -24 * norm).all()


# Matrices wide enough for tiles of 128 and 256 rows, with a last tile in each of the shorter forms: 128 + 12, 128 + 100, 256 + 43,
# 256 + 100 and 256 + 144 rows; an odd count of 64-row tiles, the last of them with 6 rows
@pytest.mark.parametrize("dtype", [8, 12, 13, 14, 30, 39])
@pytest.mark.parametrize("m", [140, 228, 299, 356, 400])
def test_full_tiles_and_a_short_last_one(dtype, m):
    from turbospark_amd import ffi
    rows, cols = 16390, 512
    rng = np.random.default_rng(m)
    entry = ffi.quantize(dtype, (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
    x = rng.standard_normal((m, cols)).astype(np.float32)
    want = x.astype(np.float16).astype(np.float64) @ ob.dequantize(dtype, entry[1], cols).astype(np.float64).T
    got = ffi.matmul(entry, x)
    # K / 16 sums in one chain (see above), by row and by column
    bound = 4 * (cols / 16) ** 0.5 * 2.0 ** -24
    for axis in (0, 1):
        assert (np.linalg.norm(got - want, axis=axis) <= bound * np.linalg.norm(want, axis=axis)).all()


def _off(entry, values, x, splits=0, column=slice(None)):
    """Distance of the prompt matmul (or one output column) from the exact product, relative to its norm."""
    from turbospark_amd import ffi
    want = (x.astype(np.float16).astype(np.float64) @ values.astype(np.float64).T)[:, column]
    return np.linalg.norm(ffi.matmul(entry, x, splits)[:, column] - want) / np.linalg.norm(want)


# Exact products summed in fp32: a sum of K = 512 values takes 32 roundings of 2^-24 of its running size, twice that where a
# weight goes in as two terms: 64^0.5 * 2^-24 = 5e-7, and one more factor of two for rows smaller than their running sums.
SUMS_OF_512 = 1e-6


@pytest.mark.parametrize("dtype", [12, 13])
@pytest.mark.parametrize("spread", ["normal", "small", "wide"])
def test_the_sums_behind_the_min_terms_keep_their_bits(dtype, spread):
    """All codes zero leaves -dmin * m * (sum of 32 activations) alone.  Sums below 1/2 are exact as the two fp16 terms they are kept
    in, larger ones to 2^-23; then two chains of two products each: 4 * 2^-24, and the same again for sums that cancel."""
    from turbospark_amd import ffi
    rng = np.random.default_rng(6)
    b = np.array(ffi.quantize(dtype, (rng.standard_normal((64, 512)) * 0.02).astype(np.float32))[1]).reshape(64, 2, -1)
    b[:, :, 16:] = 0
    entry = (dtype, np.ascontiguousarray(b.reshape(64, -1)), 64, 512)
    x = rng.standard_normal((65, 512)).astype(np.float32)
    x = x if spread == "normal" else x * 1e-3 if spread == "small" else np.sign(x) * 2.0 ** rng.uniform(-14, 4, x.shape).astype(np.float32)
    assert _off(entry, ob.dequantize(dtype, entry[1], 512), x.astype(np.float32)) <= 8 * 2.0 ** -24


@pytest.mark.parametrize("m", [17, 65, 129, 257])
@pytest.mark.parametrize("rows,at,big", [(64, 0, 2.0 ** 12), (64, 17, 2.0 ** 31), (130, 129, 2.0 ** 36), (200, 70, 2.0 ** 90), (256, 255, 3e38)])
def test_bf16_rows_of_any_span_keep_their_bits(rows, at, big, m):
    """One value far above the rest of a row, against an activation of zero: what is left are the products of the small values,
    multiplied as bf16 where they are no normal fp16 beside that one (2^29 below it), in the tiles it concerns."""
    from turbospark_amd import ffi
    rng = np.random.default_rng(rows + m)
    w, x = (rng.standard_normal((rows, 512)) * 0.02).astype(np.float32), rng.standard_normal((m, 512)).astype(np.float32)
    w[at, 7] = big
    w[rows // 2, 100] = 1e-39                          # and one with a subnormal value
    x[:, 7] = 0.0
    entry = ffi.quantize(ffi.BF16, w)
    values = (np.asarray(entry[1]).reshape(rows, -1).view(np.uint16).astype(np.uint32) << 16).view(np.float32)
    for splits in (0, 1):
        assert _off(entry, values, x, splits) <= SUMS_OF_512
        assert _off(entry, values, x, splits, at) <= SUMS_OF_512


@pytest.mark.parametrize("dtype,scale", [(39, 127), (39, 170), (39, 254), (8, 1.0), (8, 65504.0)])
def test_a_zero_block_of_any_scale_is_zero(dtype, scale):
    """Blocks whose codes are all zero do not set the power of two that their row is multiplied in."""
    from turbospark_amd import ffi
    rng = np.random.default_rng(3)
    entry = ffi.quantize(dtype, (rng.standard_normal((64, 512)) * 0.02).astype(np.float32))
    head = 1 if dtype == 39 else 2
    b = np.array(entry[1]).reshape(64, 16, -1)
    b[:, 0] = 0
    values = ob.dequantize(dtype, np.ascontiguousarray(b.reshape(64, -1)), 512)
    b[:, 0, :head] = np.frombuffer(np.uint8(scale).tobytes() if dtype == 39 else np.float16(scale).tobytes(), np.uint8)
    entry = (dtype, np.ascontiguousarray(b.reshape(64, -1)), 64, 512)
    assert _off(entry, values, rng.standard_normal((65, 512)).astype(np.float32)) <= SUMS_OF_512


@pytest.mark.parametrize("scale,rest,held", [(0.125, 2.0 ** -24, True), (0.25, 2.0 ** -24, False), (0.25, 1.99 * 2.0 ** -23, True),
                                             (65504.0, 2.0 ** -6, True), (65504.0, 2.0 ** -7, False), (np.inf, 1.0, False)])
def test_q8_0_scales_keep_their_bits_or_the_product_is_refused(scale, rest, held):
    """Scales down to 2^21 below the row's largest; a row with a smaller one is not multiplied in fp16."""
    from turbospark_amd import ffi
    rng = np.random.default_rng(4)
    b = np.array(ffi.quantize(8, (rng.standard_normal((64, 512)) * 0.02).astype(np.float32))[1]).reshape(64, 16, 34)
    b[:, 0, :2] = np.frombuffer(np.float16(scale).tobytes(), np.uint8)
    b[:, 1:, :2] = np.frombuffer(np.float16(rest).tobytes(), np.uint8)
    entry = (8, np.ascontiguousarray(b.reshape(64, -1)), 64, 512)
    x = rng.standard_normal((65, 512)).astype(np.float32)
    x[:, :32] = 0.0
    if held:
        assert _off(entry, ob.dequantize(8, entry[1], 512), x) <= SUMS_OF_512
    else:
        with pytest.raises(ffi.TsvError):
            ffi.matmul(entry, x)


@pytest.mark.parametrize("low,held", [(127 - 25, True), (127 - 26, False), (255, False)])
def test_mxfp4_blocks_keep_their_bits_or_the_product_is_refused(low, held):
    from turbospark_amd import ffi
    rng = np.random.default_rng(5)
    b = np.array(ffi.quantize(39, rng.standard_normal((64, 512)).astype(np.float32))[1]).reshape(64, 16, 17)
    b[:, 0, 0], b[:, 1:, 0] = 127, low
    entry = (39, np.ascontiguousarray(b.reshape(64, -1)), 64, 512)
    x = rng.standard_normal((65, 512)).astype(np.float32)
    x[:, :32] = 0.0
    if held:
        assert _off(entry, ob.dequantize(39, entry[1], 512), x) <= SUMS_OF_512
    else:
        with pytest.raises(ffi.TsvError):
            ffi.matmul(entry, x)


@pytest.mark.parametrize("name", ["tiny_q8_0", "gptoss_small"])
def test_a_model_of_rows_that_fp16_cannot_hold_prompts_as_before(name):
    """The first 32 columns of the query, key and value projections hold weights 2^30 above the others (behind a norm weight of
    zero): a Q8_0 model takes the smaller passes, a bf16 one multiplies those tiles as bf16."""
    from turbospark_amd import ffi, synth
    n = 100
    cfg = dict(synth.CONFIGS[name], max_context=n + 32)
    w = synth.make_weights(cfg, seed=8)
    for lw in w["layers"]:
        _, v, r, c = lw["attn_norm"]
        v = np.array(v)
        v.view(np.float32)[0, :32] = 0.0
        lw["attn_norm"] = (ffi.F32, v, r, c)
        for key in ("wq", "wk", "wv"):
            dt, v, r, c = lw[key]
            v = np.array(v)
            if dt == ffi.Q8_0:
                b = v.reshape(r, -1, 34)
                b[:, 0, :2], b[:, 0, 2:] = np.frombuffer(np.float16(2.0 ** 15).tobytes(), np.uint8), 1
            else:
                v.reshape(r, -1).view(np.uint16)[:, :32] = np.float32(2.0 ** 30).view(np.uint32) >> 16
            lw[key] = (dt, v, r, c)
    fast, slow = gc.engine(cfg, w, "prompt"), gc.engine(cfg, w, "16")
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for eng in (fast, slow):
        eng.prefill(prompt, 0, want_logits=False)
    assert gc.took(fast, "64" if name == "tiny_q8_0" else "prompt") and gc.took(slow, "16")
    for got, want in zip(fast.read_kv(0, 0, n), slow.read_kv(0, 0, n)):
        got, want = got.astype(np.float32), want.astype(np.float32)
        # each side rounds an fp32 sum to fp16: two units in the last place of the largest value
        assert np.abs(got - want).max() <= 2 * 2.0 ** -11 * np.abs(want).max()


@pytest.mark.parametrize("nq,nkv,hd", [(8, 8, 64), (32, 8, 128), (16, 2, 64), (6, 2, 128)])
@pytest.mark.parametrize("m,base,window,sinks", [(17, 0, 0, False), (33, 15, 0, True), (64, 200, 24, False), (130, 1000, 128, True),
                                                 (70, 3001, 0, True), (300, 5, 40, False)])
def test_prompt_attention_matches_the_oracle(nq, nkv, hd, m, base, window, sinks):
    from turbospark_amd import ffi
    rng = np.random.default_rng(m + base)
    r16 = lambda *s: rng.standard_normal(s).astype(np.float16).astype(np.float32)
    q, k, v = r16(m, nq, hd), r16(base + m, nkv, hd), r16(base + m, nkv, hd)
    sk = rng.standard_normal(nq).astype(np.float32) if sinks else None
    got = ffi.attention(q, k, v, base, window=window, sinks=sk)
    rows = sorted({0, 1, 15, 16, m // 2, m - 2, m - 1})
    for i in rows:
        want = ob.causal_attention(q[i], k, v, hd, nq, nkv, base + i + 1, window, 0.0, sk).reshape(nq, hd)
        assert np.abs(got[i] - want).max() <= 5e-3 * max(1.0, np.abs(want).max()), i   # the bound of the verify passes' test


@pytest.mark.parametrize("nq,nkv,hd", [(8, 8, 64), (16, 4, 128)])
@pytest.mark.parametrize("end", [991, 992, 1503, 1504, 8200])   # one chunk of the context, two, two, three, sixteen
def test_prompt_attention_at_the_lines_of_its_chunks(nq, nkv, hd, end):
    from turbospark_amd import ffi
    m = 40
    rng = np.random.default_rng(end)
    r16 = lambda *s: rng.standard_normal(s).astype(np.float16).astype(np.float32)
    q, k, v = r16(m, nq, hd), r16(end, nkv, hd), r16(end, nkv, hd)
    sk = rng.standard_normal(nq).astype(np.float32) if end % 2 else None
    got = ffi.attention(q, k, v, end - m, sinks=sk)
    for i in (0, 17, m - 1):
        want = ob.causal_attention(q[i], k, v, hd, nq, nkv, end - m + i + 1, 0, 0.0, sk).reshape(nq, hd)
        assert np.abs(got[i] - want).max() <= 5e-3 * max(1.0, np.abs(want).max()), i


@pytest.mark.parametrize("nq,nkv,hd", [(8, 2, 128), (4, 2, 64)])
@pytest.mark.parametrize("m,base,spread", [(320, 0, 1.0), (320, 0, 2.5), (96, 2000, 1.0), (96, 2000, 2.5)])
def test_prompt_attention_is_the_exact_result_rounded(nq, nkv, hd, m, base, spread):
    """Against softmax and product in 64 bits: the distance is that of the exact result rounded to fp16.  Weights of 21 bits and
    fp32 sums add a part in 2^-9 of that rounding and less; one per cent covers what is left of it by chance, 1e-5 the scores'
    own fp32 sums (128 products of a few units: 2^-24 of about 50, seen through exp)."""
    from turbospark_amd import ffi
    rng = np.random.default_rng(m + base)
    r16 = lambda *s: rng.standard_normal(s).astype(np.float16).astype(np.float32)
    q = (r16(m, nq, hd) * spread).astype(np.float16).astype(np.float32)
    k, v = r16(base + m, nkv, hd), r16(base + m, nkv, hd)
    want = np.empty((m, nq, hd))
    hidden = np.arange(base + m)[None] > base + np.arange(m)[:, None]
    for h in range(nq):
        s = q[:, h].astype(np.float64) @ k[:, h * nkv // nq].astype(np.float64).T / np.sqrt(hd)
        s[hidden] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want[:, h] = (p / p.sum(1, keepdims=True)) @ v[:, h * nkv // nq].astype(np.float64)
    got = np.asarray(ffi.attention(q, k, v, base)).reshape(m, nq, hd)
    off = lambda t: np.linalg.norm(t - want) / np.linalg.norm(want)
    assert off(got) <= 1.01 * off(want.astype(np.float16).astype(np.float64)) + 1e-5


@pytest.mark.parametrize("name,n,start", [("small_q4_k", 65, 0), ("xcd_q8_0", 257, 3), ("small_q5_k_m", 300, 31), ("xcd_q4_k", 2049, 0)])
def test_prompts_around_the_limits_of_a_pass(name, n, start):
    """Logits of the last token, what a verify pass after the prompt sees, and the rows left for tsv_accept, against passes of
    sixteen rows."""
    import turbospark_amd as ts
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS[name], max_context=start + n + 32)
    w = synth.make_weights(cfg, seed=3)
    fast, slow = gc.engine(cfg, w, "prompt"), gc.engine(cfg, w, "16")
    rng = np.random.default_rng(n)
    prompt = rng.integers(0, cfg["vocab"], start + n).astype(np.int32)
    feed = rng.integers(0, cfg["vocab"], 5).astype(np.int32)
    out = []
    for eng in (fast, slow):
        if start:
            eng.prefill(prompt[:start], 0, want_logits=False)
        last = eng.prefill(prompt[start:], start)
        m = (n - 1) % 16 + 1
        acc = eng.accept(prompt[start + n - m:], start + n - m, ts.shaping(0.0))
        eng.reset()
        eng.prefill(prompt, 0, want_logits=False)
        out.append((last, eng.verify(feed, start + n), acc))
    assert gc.took(fast, "prompt") and gc.took(slow, "16")
    assert gc.logit_error(out[0][0].reshape(1, -1), out[1][0].reshape(1, -1)) <= 2e-3
    assert gc.logit_error(out[0][1], out[1][1]) <= 2e-3
    assert (out[0][2].accepted, out[0][2].kv_position) == (out[1][2].accepted, out[1][2].kv_position)


# members of an expert around the 32- and 64-row blocks of its tiles (n * top_k / experts: 16 to 95 in tiles of 64, 125 and 250 above)
@pytest.mark.parametrize("name,n", [("moe_small", 64), ("moe_small", 129), ("moe_small", 250), ("moe_small", 383), ("moe_small", 500),
                                    ("gptoss_small", 65), ("gptoss_small", 130), ("gptoss_small", 190), ("gptoss_small", 500)])
def test_routed_prompts_give_every_row_its_experts(name, n):
    """The second layer's K and V rows, which the first layer's experts made, against passes of sixteen rows.  Single rows may
    differ where a last expert falls the other way (one decision in two hundred lies within the rounding of a tie); a wrong
    block edge would move a row of every expert, a tenth of all rows and more."""
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS[name], max_context=n + 32)
    w = synth.make_weights(cfg, seed=5)
    fast, slow = gc.engine(cfg, w, "prompt"), gc.engine(cfg, w, "16")
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for eng in (fast, slow):
        eng.prefill(prompt, 0, want_logits=False)
    assert gc.took(fast, "prompt" if n > 64 else "64") and gc.took(slow, "16")
    for got, want in zip(fast.read_kv(1, 0, n), slow.read_kv(1, 0, n)):
        got, want = got.astype(np.float32).reshape(n, -1), want.astype(np.float32).reshape(n, -1)
        # 8 units in the last place of an fp16 value of the row's largest size: fp32 sums in another order, rounded to fp16 activations
        far = np.abs(got - want).max(1) > 8 * 2.0 ** -11 * np.abs(want).max(1)
        assert far.sum() <= max(1, n // 50), np.flatnonzero(far)


# the most experts and the most pairs of a pass, every expert chosen by every row (runs without a padded block, no block past the
# last), few pairs for many experts (most blocks lie past the last run); an odd count for the last block's filling
@pytest.mark.parametrize("experts,top_k,n", [(256, 8, 2048), (8, 8, 2048), (256, 8, 97), (3, 1, 81), (1, 1, 96)])
def test_routed_prompts_at_the_limits_of_the_sort(experts, top_k, n):
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS["moe_small"], max_context=n + 32, n_experts=experts, top_k=top_k)
    w = synth.make_weights(cfg, seed=5)
    fast, slow = gc.engine(cfg, w, "prompt"), gc.engine(cfg, w, "16")
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for eng in (fast, slow):
        eng.prefill(prompt, 0, want_logits=False)
    assert gc.took(fast, "prompt") and gc.took(slow, "16")
    for got, want in zip(fast.read_kv(1, 0, n), slow.read_kv(1, 0, n)):
        got, want = got.astype(np.float32).reshape(n, -1), want.astype(np.float32).reshape(n, -1)
        far = np.abs(got - want).max(1) > 8 * 2.0 ** -11 * np.abs(want).max(1)   # as above
        assert far.sum() <= max(1, n // 50), np.flatnonzero(far)


# experts in every storage type: with sums (Q4_K, Q5_K: of the gathered rows, and of what gate / up leave), without, and mixed;
# 16 experts of which four are chosen, 21 to 94 members an expert (tiles of 64 rows) and 188 (128)
@pytest.mark.parametrize("expert,down", [(12, 12), (13, 14), (14, 13), (8, 8), (30, 30), (12, 8), (39, 12)])
@pytest.mark.parametrize("n", [84, 375, 750])
def test_routed_prompts_in_every_storage_type(expert, down, n):
    from turbospark_amd import ffi, synth
    cfg = dict(synth.CONFIGS["moe_small"], max_context=n + 32, expert_dtype=expert)
    w = synth.make_weights(cfg, seed=5)
    for lw in w["layers"]:
        lw["we_down"] = ffi.synth_tensor(down, 5, 900, 0.02, lw["we_down"][2], lw["we_down"][3])
    fast, slow = gc.engine(cfg, w, "prompt"), gc.engine(cfg, w, "16")
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for eng in (fast, slow):
        eng.prefill(prompt, 0, want_logits=False)
    assert gc.took(fast, "prompt") and gc.took(slow, "16")
    for got, want in zip(fast.read_kv(1, 0, n), slow.read_kv(1, 0, n)):
        got, want = got.astype(np.float32).reshape(n, -1), want.astype(np.float32).reshape(n, -1)
        far = np.abs(got - want).max(1) > 8 * 2.0 ** -11 * np.abs(want).max(1)   # as above
        assert far.sum() <= max(1, n // 50), np.flatnonzero(far)


@pytest.mark.parametrize("dtype,n", [(12, 100), (8, 300)])
def test_rows_wider_than_a_waves_registers(dtype, n):
    """Hidden 4352: the norm reads such a row twice (shapes of 70B models are 8192 wide).  K and V rows of both layers against
    passes of sixteen rows."""
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS["xcd_q4_k"], hidden=4352, n_q_heads=8, n_kv_heads=2, ffn=512, dtype=dtype, max_context=n + 32)
    w = synth.make_weights(cfg, seed=6)
    fast, slow = gc.engine(cfg, w, "prompt"), gc.engine(cfg, w, "16")
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for eng in (fast, slow):
        eng.prefill(prompt, 0, want_logits=False)
    assert gc.took(fast, "prompt") and gc.took(slow, "16")
    for layer in range(2):
        for got, want in zip(fast.read_kv(layer, 0, n), slow.read_kv(layer, 0, n)):
            got, want = got.astype(np.float32), want.astype(np.float32)
            assert np.abs(got - want).max() <= 8 * 2.0 ** -11 * np.abs(want).max()   # the bound of the routed rows


# calls of one 64-row pass, of two smaller passes and of three (prompt_pays in prefill.hip); few_experts: 65 rows give each of 100
# experts two or three
@pytest.mark.parametrize("name,n,start,logits,passes", [
    ("small_q4_k", 64, 0, False, "64"), ("small_q4_k", 64, 0, True, "16"), ("small_q4_k", 65, 0, False, "prompt"), ("small_q4_k", 80, 0, True, "prompt"),
    ("small_q4_k", 65, 4096, False, "64"), ("small_q4_k", 80, 4096, False, "prompt"), ("small_q4_k", 81, 4096, False, "prompt"),
    ("xcd_q8_0", 64, 0, False, "64"), ("xcd_q8_0", 65, 0, False, "64"), ("xcd_q8_0", 80, 0, True, "64"), ("xcd_q8_0", 81, 0, False, "prompt"),
    ("xcd_q8_0", 128, 0, False, "64"), ("xcd_q8_0", 128, 0, True, "prompt"), ("small_q4_k", 128, 0, False, "prompt"),
    ("moe_small", 65, 0, False, "prompt"), ("few_experts", 65, 0, False, "64"), ("few_experts", 80, 0, False, "prompt"), ("few_experts", 81, 0, False, "prompt")])
def test_a_call_takes_the_faster_passes(name, n, start, logits, passes):
    """Whether it does is a matter of the measurements beside the rule; here that the rule is the one they were taken for."""
    import turbospark_amd as ts
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS["moe_small" if name == "few_experts" else name], max_context=start + n + 32)
    if name == "few_experts":
        cfg["n_experts"] = 100
    eng = ts.HipVerifier(cfg, synth.make_weights(cfg, seed=2))
    if start:
        eng.prefill(np.zeros(start, np.int32), 0, want_logits=False)
    before = gc.prompt_buffers(eng)
    eng.prefill(np.arange(n, dtype=np.int32), start, want_logits=logits)
    after = gc.prompt_buffers(eng)
    assert eng.position == start + n
    assert (after[2] > before[2], after[3] > before[3]) == (passes == "prompt", passes == "64")


# the limits leave no prompt pass at all, or one of 256 rows where the context asks for 512
@pytest.mark.parametrize("name,n,limit,most,passes", [("small_q4_k", 300, 0, 0, 0), ("moe_small", 130, 1 << 20, 0, 0), ("small_q4_k", 66, 3 << 20, 0, 0),
                                                      ("small_q4_k", 300, "half", 256, 2), ("moe_small", 300, "half", 256, 2)])
def test_a_device_without_room_for_prompt_buffers_takes_smaller_passes(name, n, limit, most, passes):
    """The same call succeeds, in the passes the handle has buffers for, and takes the large passes again once there is room."""
    import turbospark_amd as ts
    from turbospark_amd import ffi, synth
    cfg = dict(synth.CONFIGS[name], max_context=n + 32)
    eng = ts.HipVerifier(cfg, synth.make_weights(cfg, seed=9))
    whole, held = gc.prompt_buffers(eng)[:2]
    assert whole == -(-(n + 32) // 256) * 256 and held > 0
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    kv = []
    for bytes_, rows, count in ((limit, most, passes), (limit, most, passes), (1 << 40, whole, 1)):
        eng.reset()
        ffi.check(ffi.lib().tsv_limit_prompt_buffers(eng._h, held - 1 if bytes_ == "half" else bytes_))
        before = gc.prompt_buffers(eng)
        eng.prefill(prompt, 0, want_logits=False)
        after = gc.prompt_buffers(eng)
        assert eng.position == n and after[:2] == (rows, held) and after[2] - before[2] == count
        assert (after[3] > before[3]) == (count == 0)
        kv.append(eng.read_kv(0, 0, n))
    for (a, b, c) in zip(*kv):          # the first layer's rows: sums of the same products
        a, b, c = (t.astype(np.float32) for t in (a, b, c))
        assert (a == b).all()
        # each side rounds an fp32 sum of about sqrt(K) roundings to fp16: two units in the last place of the largest value
        assert np.abs(a - c).max() <= 2 * 2.0 ** -11 * np.abs(a).max()


@pytest.mark.parametrize("name", ["small_q4_k", "moe_small"])
def test_prompts_of_any_length_allocate_nothing(name):
    """A handle's buffers come with it: the device's free memory is the same before and after prompts that grow."""
    import ctypes as C
    import turbospark_amd as ts
    from turbospark_amd import hip, synth

    def room():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.rt().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    cfg = dict(synth.CONFIGS[name], max_context=2300)
    eng = ts.HipVerifier(cfg, synth.make_weights(cfg, seed=9))
    assert gc.prompt_buffers(eng)[0] == 2048
    eng.prefill(np.zeros(20, np.int32), 0, want_logits=False)     # code objects, the runtime's own first use
    free = room()
    for n in (100, 700, 2200):
        eng.reset()
        eng.prefill(np.zeros(n, np.int32), 0, want_logits=False)
        assert room() == free, n
