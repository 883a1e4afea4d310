"""Acceptance on scores no model would hand over: flat rows, two-valued rows, heavy ties, spreads that
underflow every exponential but one, the fp16 extremes, subnormals and signed zeros, tiny and odd
vocabularies.  The target rows are written to the device directly (`tsv_write_logits`), so the whole
round -- statistics, truncation cuts, the acceptance walk, residual and bonus draws, penalties, tree
walks -- is compared with the oracle's restatement of crates/runtime/src/speculative.rs:694-754,
861-879 and crates/selection/src/choose.rs:111-338, integers equal.

A case whose smallest decision margin the device itself reports below 1e-9 is not compared (a
comparison that close may legitimately fall the other way against host libm / summation order); such
cases must stay rare."""
import numpy as np
import pytest

from oracle import binding as ob
from tests import gpu_common as gc

pytestmark = pytest.mark.gpu

F16_MAX = 65504.0


def _row(r, V, kind):
    if kind == "flat":
        return np.full(V, float(r.choice([0.0, -3.5, 11.0])), np.float32)
    if kind == "two":
        a, b = r.choice([-2.0, 0.0, 0.5, 3.0, 8.0], 2, replace=False)
        return np.where(r.random(V) < r.uniform(0.01, 0.6), a, b).astype(np.float32)
    if kind == "ties":
        q = float(r.choice([1, 2, 4, 8]))
        return (np.round(r.standard_normal(V) * 2 * q) / q).astype(np.float32)
    if kind == "wide":
        return np.clip(r.standard_normal(V) * 3000.0, -F16_MAX, F16_MAX).astype(np.float32)
    if kind == "extremes":
        x = np.full(V, -F16_MAX, np.float32)
        x[r.integers(0, V, max(1, V // 50))] = F16_MAX
        x[r.integers(0, V, max(1, V // 50))] = float(r.choice([0.0, 60000.0, F16_MAX - 32.0]))
        return x
    if kind == "tiny":
        x = (r.integers(-6, 7, V) * 5.96e-8).astype(np.float32)          # fp16 subnormals around zero
        x[r.random(V) < 0.3] = -0.0
        return x
    if kind == "peaked":
        x = r.standard_normal(V).astype(np.float32)
        x[r.integers(0, V)] += float(r.choice([12.0, 30.0, 200.0]))
        return x
    return (r.standard_normal(V) * 2).astype(np.float32)


KINDS = ["flat", "two", "ties", "wide", "extremes", "tiny", "peaked", "normal"]


def _shaping(r, seed, penalties):
    import turbospark_amd as ts
    kw = {}
    if r.integers(0, 2):
        kw["top_k"] = int(r.integers(1, 257))
    if r.integers(0, 2):
        kw["top_p"] = float(r.uniform(0.05, 1.0))
    if r.integers(0, 2):
        kw["min_p"] = float(r.uniform(1e-4, 0.5))
    if penalties and r.integers(0, 2):
        kw["repetition_penalty"] = float(r.uniform(0.5, 2.0))
    if penalties and r.integers(0, 2):
        kw["presence_penalty"] = float(r.uniform(-2.0, 2.0))
        kw["frequency_penalty"] = float(r.uniform(-2.0, 2.0))
    t = float(r.choice([0.05, 0.3, 0.8, 1.0, 1.7, 4.0]))
    return ts.shaping(t, seed=seed, **kw), ob.shaping(t, seed=seed, **kw), kw


@pytest.mark.parametrize("vocab", [4096, 1000, 37, 2, 128256, 201088])
def test_adversarial_chain_rounds(vocab):
    """(128256 and 201088: the vocabularies of the benchmark configurations, fewer and narrower rounds.)"""
    cfg, w, gpu, cpu = gc.build_pair("tiny_q8_0", max_context=64, vocab=vocab)
    V = vocab
    r = np.random.default_rng(77 + vocab)
    base = 20
    compared = skipped = 0
    outcomes = set()
    big = V > 100000
    for case in range(14 if big else 60):
        k = int(r.integers(0, 6 if big else 16))
        kind_t, kind_d = r.choice(KINDS), r.choice(KINDS)
        target = np.stack([_row(r, V, kind_t) for _ in range(k + 1)]).astype(np.float16)
        # the drafter: adversarial rows of its own, or the target's rows nudged (so that proposals get accepted)
        if r.integers(0, 2) and k:
            draft = (target[:k].astype(np.float32) + (r.standard_normal((k, V)) * 0.05).astype(np.float32)).astype(np.float16)
        else:
            draft = np.stack([_row(r, V, kind_d) for _ in range(max(k, 1))]).astype(np.float16)[:max(k, 1)]
        # (a penalised score below every fp16 value is refused by name: no penalties on the rows that sit there)
        gcfg, ocfg, kw = _shaping(r, 100 + case, penalties=not {kind_t, kind_d} & {"wide", "extremes"})
        hist = [int(t) for t in r.integers(-2, V + 2, int(r.integers(0, 300)))]
        generated = int(r.integers(0, len(hist) + 2))
        ds = int(r.integers(0, 1000))
        stops = [int(t) for t in r.integers(0, V, int(r.integers(0, 3)))]
        budget = generated + int(r.integers(1, 20))
        try:
            if k:
                props, ds1 = gpu.draft_chain(draft[:k], gcfg, ds, history=hist, generated=generated)
                oprops, ods1 = ob.draft_chain(draft[:k], ocfg, hist, generated, ds)
            else:
                props, ds1, oprops, ods1 = np.zeros(0, np.int32), ds, np.zeros(0, np.int32), ds
        except Exception as e:  # a refusal by name (more penalised candidates in one rank bin than the list holds)
            assert "not built" in str(e), e
            skipped += 1
            continue
        feed = [int(r.integers(0, V))] + [int(t) for t in oprops]
        gpu.write_logits(target, base)
        try:
            res = gpu.accept(feed, base, gcfg, draft_logits=draft, draw_step=ods1, stop_tokens=stops, generated=generated,
                             max_new_tokens=budget, history=hist)
        except Exception as e:
            assert "not built" in str(e), e
            skipped += 1
            continue
        want = ob.chain_round(target.view(np.uint16), draft.view(np.uint16)[:k] if k else np.zeros((0, V), np.uint16), oprops, ocfg,
                              history=hist, generated=generated, max_new_tokens=budget, stop_tokens=stops, draw_step=ods1)
        if res.min_margin < 1e-9:
            skipped += 1
            continue
        assert list(props) == list(oprops) and ds1 == ods1, (case, kind_d, kw)
        got = (res.accepted, res.committed, res.next, res.stopped, res.draw_step)
        assert got == (want["accepted"], want["committed"], want["next"], want["stopped"], want["draw_step"]), \
            (case, kind_t, kind_d, k, kw, res, want)
        assert res.kv_position == base + want["committed"] + 1
        compared += 1
        outcomes.add((res.accepted == k, res.stopped))
    print(f"vocab {vocab}: {compared} rounds compared, {skipped} too close to call or refused by name; outcomes {sorted(outcomes)}")
    assert compared >= (10 if big else 45) and len(outcomes) >= 2


@pytest.mark.parametrize("vocab", [4096, 333])
def test_adversarial_tree_rounds(vocab):
    cfg, w, gpu, cpu = gc.build_pair("tiny_q8_0", max_context=64, vocab=vocab)
    V = vocab
    r = np.random.default_rng(5 + vocab)
    base = 20
    compared = skipped = 0
    for case in range(40):
        m = int(r.integers(2, 17))
        parent = [-1] + [int(r.integers(0, s)) for s in range(1, m)]
        kind_t, kind_d = r.choice(KINDS), r.choice(KINDS)
        target = np.stack([_row(r, V, kind_t) for _ in range(m)]).astype(np.float16)
        if r.integers(0, 2):
            draft = (target.astype(np.float32) + (r.standard_normal((m, V)) * 0.05).astype(np.float32)).astype(np.float16)
        else:
            draft = np.stack([_row(r, V, kind_d) for _ in range(m)]).astype(np.float16)
        feed = [int(t) for t in r.integers(0, V, m)]
        # children drawn from where the mass is, so that walks go deep
        for s in range(1, m):
            if r.integers(0, 2):
                feed[s] = int(np.argmax(target[parent[s]].astype(np.float32) + r.standard_normal(V) * 0.5))
        sampled = bool(r.integers(0, 4))
        gcfg, ocfg, kw = _shaping(r, 300 + case, penalties=not {kind_t, kind_d} & {"wide", "extremes"})
        if not sampled:
            import turbospark_amd as ts
            gcfg, ocfg = ts.shaping(0.0), ob.shaping(0.0)
        hist = [int(t) for t in r.integers(0, V, int(r.integers(0, 200)))]
        generated = int(r.integers(0, len(hist) + 2))
        gpu.write_logits(target, base)
        try:
            res = gpu.accept(feed, base, gcfg, parent=parent, draft_logits=draft if sampled else None, draw_step=9,
                             history=hist, generated=generated)
        except Exception as e:
            assert "not built" in str(e), e
            skipped += 1
            continue
        if sampled:
            want = ob.tree_round_sampled(target.view(np.uint16), draft.view(np.uint16), feed, parent, ocfg, history=hist,
                                         generated=generated, draw_step=9)
        else:
            want = ob.tree_round_greedy(target.view(np.uint16), feed, parent, ocfg, history=hist)
        if res.min_margin < 1e-9:
            skipped += 1
            continue
        assert res.path == want["path"] and res.next == want["next"], (case, kind_t, kind_d, kw, res, want)
        if sampled:
            assert res.draw_step == want["draw_step"]
        compared += 1
    print(f"vocab {vocab}: {compared} tree rounds compared, {skipped} too close to call or refused by name")
    assert compared >= 30


@pytest.mark.parametrize("vocab", [40, 1000, 4096])
@pytest.mark.parametrize("penalty", [None, 1.25])
def test_truncation_cuts_at_the_edges_of_a_group_of_rank_bins(vocab, penalty):
    """The cuts are found in two levels, groups of 64 rank bins and the bins of one: candidates in the last bin of a group, the first of the next
    one and the last bin but one group, five each (some of them reweighted by a penalty), and cuts that fall before, on and behind each
    edge, by count, by mass, and by both in one group or in two."""
    import turbospark_amd as ts
    cfg, w, gpu, cpu = gc.build_pair("tiny_q8_0", max_context=64, vocab=vocab)
    edge = np.array([0x4840, 0x4800, 0x47FF], np.uint16)          # 8.5, 8.0: key % 64 == 63; the value below 8.0: key % 64 == 0
    assert [int((0xFFFF - (int(b) | 0x8000)) % 64) for b in edge] == [63, 63, 0]
    bits = np.full(vocab, np.float16(-3.0).view(np.uint16), np.uint16)
    at = np.random.default_rng(5).permutation(vocab)[:15]
    bits[at] = np.repeat(edge, 5)
    target = bits.view(np.float16)[None]
    e = np.exp(target[0].astype(np.float64) - 8.5)
    share = np.cumsum(np.sort(e / e.sum())[::-1])
    history = [int(t) for t in at[::4]] if penalty else []
    kws = [dict(top_k=k) for k in (1, 4, 5, 6, 9, 10, 11, 14, 15, 16)]
    kws += [dict(top_p=float(0.5 * (share[i] + share[i + 1]))) for i in (0, 3, 4, 5, 8, 9, 10, 13)]
    kws += [dict(top_k=k, top_p=float(0.5 * (share[i] + share[i + 1]))) for k, i in ((10, 4), (11, 9), (6, 8), (5, 12), (15, 2))]
    compared = 0
    for n, kw in enumerate(kws):
        if penalty:
            kw = dict(kw, repetition_penalty=penalty)
        for seed in range(4):
            gcfg, ocfg = ts.shaping(1.0, seed=10 * n + seed, **kw), ob.shaping(1.0, seed=10 * n + seed, **kw)
            gpu.write_logits(target, 20)
            res = gpu.accept([3], 20, gcfg, draft_logits=np.zeros((1, vocab), np.float16), history=history)
            want = ob.chain_round(target.view(np.uint16), np.zeros((0, vocab), np.uint16), np.zeros(0, np.int32), ocfg, history=history)
            if res.min_margin < 1e-9:
                continue
            assert (res.next, res.draw_step) == (want["next"], want["draw_step"]), (kw, seed)
            compared += 1
    assert compared >= 3 * len(kws)


def _seed_drawing(bits53, position):
    """The seed whose uniform at `position` is bits53 2^-53: splitmix64's finaliser (crates/selection/src/derive.rs:19-45) undone step by step."""
    mask = (1 << 64) - 1

    def unshift(x, n):
        y = x
        for _ in range(64 // n + 1):
            y = x ^ (y >> n)
        return y
    x = unshift(bits53 << 11, 31)
    x = unshift(x * pow(0x94D049BB133111EB, -1, 1 << 64) & mask, 27)
    x = unshift(x * pow(0xBF58476D1CE4E5B9, -1, 1 << 64) & mask, 30)
    x = (x - 0x9E3779B97F4A7C15) & mask
    return x ^ (position * 0x9E3779B97F4A7C15 & mask)


@pytest.mark.parametrize("vocab", [37, 1000, 4096])
@pytest.mark.parametrize("penalty", [None, 1.25])
def test_draws_at_the_ends_of_the_uniform(vocab, penalty):
    """The smallest and the largest uniforms there are.  At the largest ones the sums in fixed point and in doubles part by a rounding, no candidate's sum
    passes the uniform and the draw takes the bin's last: plain draws and draws from a residual, against the oracle.  Rows whose last candidate carries mass enough that
    rounding cannot decide between it and the one before."""
    import turbospark_amd as ts
    cfg, w, gpu, cpu = gc.build_pair("tiny_q8_0", max_context=64, vocab=vocab)
    r = np.random.default_rng(9)
    top = (1 << 53) - 1
    for kind in ("flat", "two", "ties", "normal"):
        row = _row(r, vocab, kind).astype(np.float16)
        sure = int(np.argmin(row))                                       # the drafter proposes what the target least wants: refused
        draft = np.full((1, vocab), -8.0, np.float16)
        draft[0, sure] = 20.0
        history = [int(t) for t in r.integers(0, vocab, 30)] if penalty else []
        kw = dict(repetition_penalty=penalty) if penalty else {}
        for bits in (0, 1, top - 1, top):
            for feed, position in (([3], 0), ([3, sure], 1)):
                seed = _seed_drawing(bits, position)
                target = np.stack([row] * len(feed))
                gpu.write_logits(target, 20)
                res = gpu.accept(feed, 20, ts.shaping(1.0, seed=seed, **kw), draft_logits=draft, history=history)
                want = ob.chain_round(target.view(np.uint16), draft.view(np.uint16)[:len(feed) - 1], np.asarray(feed[1:], np.int32),
                                      ob.shaping(1.0, seed=seed, **kw), history=history)
                assert (res.accepted, res.draw_step) == (want["accepted"], want["draw_step"])
                assert res.next == want["next"], (kind, bits, feed)


@pytest.mark.parametrize("flat", [(0,), (1,), (7,), (14,), (3, 14)])
def test_a_draw_that_is_refused_is_refused_whichever_row_it_is_of(flat):
    """Rows of which 1500 penalised candidates share a score between two fp16 values, more than a draw can put in order, among rows that draw without any."""
    import turbospark_amd as ts
    vocab, k = 4096, 15
    cfg, w, gpu, cpu = gc.build_pair("tiny_q8_0", max_context=64, vocab=vocab)
    hist = list(range(1500))
    r = np.random.default_rng(5)
    rows = (r.standard_normal((k, vocab)) * 0.5).astype(np.float16)
    rows[:, 2000] = 20.0                                             # sure of a token that no penalty touches
    for seed in range(3):
        draft = rows.copy()
        gpu.draft_chain(draft, ts.shaping(1.0, seed=seed, repetition_penalty=1.1), 0, history=hist)
        draft[list(flat)] = -40.0
        draft[list(flat), :1500] = 3.0
        with pytest.raises(Exception, match="not built"):
            gpu.draft_chain(draft, ts.shaping(1.0, seed=seed, repetition_penalty=1.1), 0, history=hist)
