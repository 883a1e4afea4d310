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
    import os
    import turbospark_amd as ts
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS[name], max_context=start + n + 32)
    w = synth.make_weights(cfg, seed=3)
    fast = ts.HipVerifier(cfg, w)
    os.environ["TSV_WIDE_PREFILL"] = "0"
    try:
        slow = ts.HipVerifier(cfg, w)
    finally:
        del os.environ["TSV_WIDE_PREFILL"]
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
    import os
    import turbospark_amd as ts
    from turbospark_amd import synth
    cfg = dict(synth.CONFIGS[name], max_context=n + 32)
    w = synth.make_weights(cfg, seed=5)
    fast = ts.HipVerifier(cfg, w)
    os.environ["TSV_WIDE_PREFILL"] = "0"
    try:
        slow = ts.HipVerifier(cfg, w)
    finally:
        del os.environ["TSV_WIDE_PREFILL"]
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for eng in (fast, slow):
        eng.prefill(prompt, 0, want_logits=False)
    for got, want in zip(fast.read_kv(1, 0, n), slow.read_kv(1, 0, n)):
        got, want = got.astype(np.float32).reshape(n, -1), want.astype(np.float32).reshape(n, -1)
        # 8 units in the last place of an fp16 value of the row's largest size: fp32 sums in another order, rounded to fp16 activations
        far = np.abs(got - want).max(1) > 8 * 2.0 ** -11 * np.abs(want).max(1)
        assert far.sum() <= max(1, n // 50), np.flatnonzero(far)


@pytest.mark.parametrize("name,n,limit", [("small_q4_k", 300, 0), ("moe_small", 130, 1 << 20), ("small_q4_k", 64, 3 << 20)])
def test_a_device_without_room_for_prompt_buffers_takes_the_64_row_passes(name, n, limit):
    """The buffers refused at the first and at a later allocation: the same call succeeds, in the passes the handle has buffers
    for, and takes the large passes again once there is room."""
    import turbospark_amd as ts
    from turbospark_amd import ffi, synth
    cfg = dict(synth.CONFIGS[name], max_context=n + 32)
    eng = ts.HipVerifier(cfg, synth.make_weights(cfg, seed=9))
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    kv = []
    for bytes_ in (limit, limit, 1 << 40):
        eng.reset()
        ffi.check(ffi.lib().tsv_limit_prompt_buffers(eng._h, bytes_))
        eng.prefill(prompt, 0, want_logits=False)
        assert eng.position == n
        kv.append(eng.read_kv(0, 0, n))
    for (a, b, c) in zip(*kv):          # the first layer's rows: sums of the same products
        a, b, c = (t.astype(np.float32) for t in (a, b, c))
        assert (a == b).all()
        # each side rounds an fp32 sum of about sqrt(K) roundings to fp16: two units in the last place of the largest value
        assert np.abs(a - c).max() <= 2 * 2.0 ** -11 * np.abs(a).max()
