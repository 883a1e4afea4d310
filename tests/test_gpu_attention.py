"""GPU parity of the verify-pass attention kernel against the oracle's causal attention.

Mirrors crates/gpu/tests/attention_tree_parity.rs (identity path == chain row; a branch node ==
the chain over its root path) and crates/compute/src/attention.rs' reference arithmetic."""
import numpy as np
import pytest

from oracle import binding as ob

pytestmark = pytest.mark.gpu


def _oracle(q, k, v, base, parent, scale=0.0, window=0, sinks=None):
    m, nq, hd = q.shape
    nkv = k.shape[1]
    out = np.empty((m, nq, hd), np.float32)
    import ctypes as C
    sk = np.ascontiguousarray(sinks, np.float32) if sinks is not None else None
    for i in range(m):
        if parent is None:
            out[i] = ob.causal_attention(q[i], k, v, hd, nq, nkv, base + i + 1, window, scale, sinks).reshape(nq, hd)
        else:
            path = []
            s = i
            while s >= 0:
                path.append(base + s)
                s = parent[s]
            path = np.array(path[::-1], np.int64)
            start = 0
            if window and base + len(path) > window:   # the last `window` members of prefix + root path
                start = base + len(path) - window
                assert start <= base
            o = np.empty(nq * hd, np.float32)
            qq = np.ascontiguousarray(q[i], np.float32)
            kk = np.ascontiguousarray(k, np.float32)
            vv = np.ascontiguousarray(v, np.float32)
            ob.lib().tso_attention_core(qq.ctypes.data_as(C.c_void_p), kk.ctypes.data_as(C.c_void_p),
                                        vv.ctypes.data_as(C.c_void_p), hd, nq, nkv, C.c_int64(start), C.c_int64(base),
                                        path.ctypes.data_as(C.c_void_p), len(path), C.c_float(scale),
                                        sk.ctypes.data_as(C.c_void_p) if sk is not None else None,
                                        o.ctypes.data_as(C.c_void_p))
            out[i] = o.reshape(nq, hd)
    return out


def _rand(m, nq, nkv, hd, base, seed):
    rng = np.random.default_rng(seed)
    r16 = lambda *s: rng.standard_normal(s).astype(np.float16).astype(np.float32)
    return r16(m, nq, hd), r16(base + m, nkv, hd), r16(base + m, nkv, hd)


@pytest.mark.parametrize("nq,nkv,hd", [(8, 8, 64), (4, 1, 128), (32, 8, 128), (16, 2, 64)])
@pytest.mark.parametrize("m,base", [(1, 0), (1, 37), (4, 0), (5, 0), (8, 0), (16, 0), (5, 200), (16, 1000), (9, 15)])
def test_chain_attention_matches_the_oracle(nq, nkv, hd, m, base):
    from turbospark_amd import ffi
    q, k, v = _rand(m, nq, nkv, hd, base, 100 + m + base)
    got = ffi.attention(q, k, v, base)
    want = _oracle(q, k, v, base, None)
    err = np.abs(got - want).reshape(m, -1).max(1)
    assert err.max() <= 5e-3 * max(1.0, np.abs(want).max()), err  # Tolerance::FP16_REDUCTION


def test_tree_attention_sees_prefix_plus_root_path():
    from turbospark_amd import ffi
    parent = [-1, 0, 0, 0, 0, 1, 5, 6, 2, 8, 9, 3, 11, 12, 4, 14]
    for (nq, nkv, hd, base) in [(4, 1, 128, 37), (32, 8, 128, 300), (8, 8, 64, 0)]:
        q, k, v = _rand(16, nq, nkv, hd, base, 5)
        got = ffi.attention(q, k, v, base, parent)
        want = _oracle(q, k, v, base, parent)
        assert np.abs(got - want).max() <= 5e-3 * max(1.0, np.abs(want).max())
        # identity path == chain, bit for bit
        a = ffi.attention(q[:6], k[:base + 6], v[:base + 6], base)
        b = ffi.attention(q[:6], k[:base + 6], v[:base + 6], base, [-1, 0, 1, 2, 3, 4])
        assert np.array_equal(a, b)
        # the identity map over a branching layout must FAIL at branch nodes
        c = ffi.attention(q, k, v, base)
        assert np.abs(c[8] - want[8]).max() > 1e-2


@pytest.mark.parametrize("nq,nkv,hd", [(8, 2, 64), (32, 8, 128)])
@pytest.mark.parametrize("m,base,window", [(1, 0, 17), (5, 10, 17), (9, 200, 128), (16, 300, 24), (16, 1000, 128),
                                           (4, 130, 128), (9, 119, 128), (1, 127, 128), (1, 128, 128)])
def test_sliding_window_and_sinks_match_the_oracle(nq, nkv, hd, m, base, window):
    """crates/compute/src/attention.rs:53-137: kv_start = seq_len - window; the sink joins the
    maximum and the denominator only (it takes probability mass away from the real positions)."""
    from turbospark_amd import ffi
    q, k, v = _rand(m, nq, nkv, hd, base, 400 + m + base)
    sinks = np.random.default_rng(base).standard_normal(nq).astype(np.float32) * 2
    for sk in (None, sinks):
        got = ffi.attention(q, k, v, base, scale=0.125, window=window, sinks=sk)
        want = _oracle(q, k, v, base, None, 0.125, window, sk)
        assert np.abs(got - want).max() <= 5e-3 * max(1.0, np.abs(want).max()), (sk is None)
    plain = ffi.attention(q, k, v, base, scale=0.125)
    sunk = ffi.attention(q, k, v, base, scale=0.125, sinks=sinks + 4)
    assert np.all(np.abs(sunk).sum(-1) < np.abs(plain).sum(-1) + 1e-3)   # mass went to the sink
    if base + 1 > window:
        assert np.abs(ffi.attention(q, k, v, base, scale=0.125, window=window) - plain).max() > 1e-3


def test_tree_attention_with_a_window():
    from turbospark_amd import ffi
    parent = [-1, 0, 0, 0, 0, 1, 5, 6, 2, 8, 9, 3, 11, 12, 4, 14]
    sinks = np.linspace(-1, 1, 8).astype(np.float32)
    for base, window in [(37, 24), (300, 128), (5, 20)]:
        q, k, v = _rand(16, 8, 2, 64, base, 9)
        got = ffi.attention(q, k, v, base, parent, scale=0.125, window=window, sinks=sinks)
        want = _oracle(q, k, v, base, parent, 0.125, window, sinks)
        assert np.abs(got - want).max() <= 5e-3 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("nq,nkv,hd", [(32, 8, 128), (64, 8, 64), (32, 4, 128)])
@pytest.mark.parametrize("m,base,window", [(1, 130, 0), (5, 250, 0), (16, 370, 0), (1, 500, 0), (5, 480, 0), (16, 496, 0), (5, 3000, 128),
                                           (16, 200, 128)])
def test_rows_of_a_short_context_are_the_nearest_fp16(nq, nkv, hd, m, base, window):
    """Against 64 bits: what a row is off by comes from its last rounding.  The scores are fp32 sums of 128 exact products (2^-24 of
    their norm each, scores of up to 12 in units of log 2: 3e-6 of a weight at most), weights two fp16 terms (2^-22), so a value is off by
    less than 4e-6 before it is rounded, and the nearest fp16 (a step is 5e-4 of a value or more) is missed where the exact value
    lies that close to the middle of two: 2 * 4e-6 / 5e-4, less than one in fifty.  Weights rounded to fp16 (2e-4) miss two in five."""
    from turbospark_amd import ffi
    q, k, v = _rand(m, nq, nkv, hd, base, 77 + m + base)
    q *= 2
    got = ffi.attention(q, k, v, base, window=window)
    want = np.empty((m, nq, hd))
    for i in range(m):
        lo = max(0, base + i + 1 - window) if window else 0
        kk, vv = (np.repeat(a[lo:base + i + 1].astype(np.float64), nq // nkv, axis=1) for a in (k, v))
        s = np.einsum("hd,phd->hp", q[i].astype(np.float64), kk) / hd ** 0.5
        w = np.exp(s - s.max(1, keepdims=True))
        want[i] = np.einsum("hp,phd->hd", w / w.sum(1, keepdims=True), vv)
    big = np.abs(want) > 2.0 ** -6 * np.sqrt((want ** 2).mean())   # (a sum that cancels has fewer bits of its own)
    missed = np.mean(got.astype(np.float16)[big] != want.astype(np.float16)[big])
    assert missed <= 0.02, missed


@pytest.mark.parametrize("nq,nkv,hd", [(32, 8, 128), (64, 8, 64)])
@pytest.mark.parametrize("m", [1, 5, 16])
@pytest.mark.parametrize("end,window", [(17, 0), (127, 0), (128, 0), (129, 0), (900, 97), (900, 113), (900, 129),
                                        (511, 0), (512, 0), (513, 0), (900, 481), (900, 482), (900, 483)])
def test_both_sides_of_the_line_of_short_contexts(nq, nkv, hd, m, end, window):
    """Contexts and windows around the longest that one workgroup takes whole, and around the longest of one block to each of its waves."""
    from turbospark_amd import ffi
    base = end - m
    q, k, v = _rand(m, nq, nkv, hd, base, 31 * end + m)
    sinks = np.random.default_rng(m).standard_normal(nq).astype(np.float32) if window else None
    got = ffi.attention(q, k, v, base, window=window, sinks=sinks)
    want = _oracle(q, k, v, base, None, window=window, sinks=sinks)
    assert np.abs(got - want).max() <= 5e-3 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("nq,nkv,hd", [(7, 7, 64), (12, 6, 128), (10, 5, 64), (32, 4, 128), (4, 1, 64)])   # 36, 42, 51 and 64 chunks
@pytest.mark.parametrize("m,base", [(1, 560), (1, 1031), (2, 510), (2, 2600)])
def test_merge_of_more_than_thirty_two_chunks(nq, nkv, hd, m, base):
    """Counts on both sides of a batch of 32 chunks' end, contexts that leave the last chunks without a position, and long ones."""
    from turbospark_amd import ffi
    q, k, v = _rand(m, nq, nkv, hd, base, 7 * base + nkv)
    sinks = np.random.default_rng(nkv).standard_normal(nq).astype(np.float32) if base % 2 else None
    got = ffi.attention(q, k, v, base, sinks=sinks)
    want = _oracle(q, k, v, base, None, sinks=sinks)
    assert np.abs(got - want).max() <= 5e-3 * max(1.0, np.abs(want).max())


@pytest.mark.parametrize("seed", range(64))
def test_random_attention_shapes_and_long_contexts(seed):
    """Seeded sweep: head width, GQA group 1..8, 1..16 rows, chain or random tree, contexts up to 20000
    positions (several 16-position blocks per wave: the pipelined walk), optional window (wider than
    the pass) and sinks, a scale of its own."""
    from turbospark_amd import ffi
    r = np.random.default_rng(4000 + seed)
    hd = int(r.choice([64, 128]))
    nkv = int(r.choice([1, 2, 4, 8]))
    g = int(r.choice([1, 2, 3, 4, 8]))
    nq = nkv * g
    m = int(r.integers(1, 17))
    base = int(r.choice([0, 1, 15, 16, 17, int(r.integers(18, 600)), int(r.integers(600, 5000)), int(r.integers(5000, 20000))]))
    tree = bool(r.integers(0, 2)) and m > 2
    parent = [-1] + [int(r.integers(0, s)) for s in range(1, m)] if tree else None
    window = int(r.integers(17, 300)) if r.integers(0, 3) == 0 else 0
    sinks = (r.standard_normal(nq) * 2).astype(np.float32) if r.integers(0, 3) == 0 else None
    scale = float(r.choice([0.0, 0.1, 0.2]))
    q, k, v = _rand(m, nq, nkv, hd, base, 9000 + seed)
    print(f"seed {seed}: hd={hd} q/kv={nq}/{nkv} m={m} base={base} {'tree' if tree else 'chain'} window={window} "
          f"sinks={'yes' if sinks is not None else 'no'} scale={scale}", flush=True)
    got = ffi.attention(q, k, v, base, parent=parent, scale=scale, window=window, sinks=sinks)
    want = _oracle(q, k, v, base, parent, scale=scale, window=window, sinks=sinks)
    err = np.abs(got - want).max()
    assert err <= 5e-3 * max(1.0, np.abs(want).max()), err
