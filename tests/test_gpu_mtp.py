"""The drafter head inside the library (docs/MTP.md:53-60, crates/runtime/src/families/qwen/mtp.rs) against the
oracle's restatement of the recurrence, and the loop's block-draft and chunked-prefill callbacks
(producer.rs:193-250) against the token-at-a-time, step-by-step walk of the same head."""
import numpy as np
import pytest

import turbospark_amd as ts
from oracle import binding as ob
from tests import gpu_common as gc
from tests.loop_common import GpuTarget
from turbospark_amd import ffi, synth

pytestmark = pytest.mark.gpu

KEYS = ("tokens", "stop_reason", "rounds", "offered", "accepted", "rollbacks", "draw_step", "final_depth")


def _build(name, ctx=160, oracle=True, **over):
    cfg = dict(synth.CONFIGS[name], max_context=ctx)
    cfg.update(over)
    w = synth.make_weights(cfg, seed=1234)
    hcfg, hw = synth.make_mtp_weights(cfg, w, seed=77, follow=over.get("follow", 0.0))
    gpu = ts.HipVerifier(cfg, w)
    head = ts.MtpHead(gpu, hcfg, hw)
    if not oracle:
        return cfg, gpu, head
    return cfg, gpu, head, ob.Model(cfg, w, threads=8), ob.MtpHead(hcfg, hw, threads=8)


def _amax(bits):
    return int(np.argmax(gc.f16(bits)))


@pytest.mark.parametrize("name", ["tiny_q8_0", "small_q4_k", "xcd_q4_k", "moe_small", "gptoss_small"])
def test_the_heads_logits_match_the_oracle_through_priming_steps_chained_steps_and_a_rewind(name):
    cfg, gpu, head, trunk, ohead = _build(name)
    V = cfg["vocab"]
    tol = gc.TOL.get(cfg["dtype"], 1e-2)
    prompt = np.random.default_rng(4).integers(0, V, 21).astype(np.int32)
    n = len(prompt)
    # the prompt: the target's prefill primes the head over every position whose next token is known
    last = head.prefill_chunk(prompt, 0)
    want_last = trunk.verify(prompt, 0)[-1]
    assert gc.logit_error(last, want_last) <= tol
    ohead.step(prompt[1:], np.array([trunk.last_hidden(r) for r in range(n - 1)]), 0, want=None)
    assert head.position == n - 1 == ohead.position
    k_got, v_got = head.read_kv(0, n - 1)
    k_want, v_want = ohead.model.kv(0)
    assert np.abs(k_got.astype(np.float32).reshape(n - 1, -1) - k_want[:n - 1].reshape(n - 1, -1)).max() <= 3e-2
    # a round: the step from the target's state, two chained steps from the head's own
    nxt = _amax(want_last)
    base = n
    got = head.step(nxt, base - 1)
    want = ohead.step([nxt], trunk.last_hidden(n - 1), base - 1)[0]
    errs = [gc.logit_error(got, want)]
    feed = [nxt]
    for d in (1, 2):
        tok = _amax(want)
        feed.append(tok)
        got = head.step(tok, base - 1 + d)
        want = ohead.step([tok], ohead.last_hidden(0), base - 1 + d)[0]
        errs.append(gc.logit_error(got, want))
    # the target verifies the three tokens; say one proposal was committed: both heads go back to base + 1
    gpu.verify(feed, base, want_logits=False)
    trunk.verify(feed, base)
    head.rewind(base + 1)
    ohead.rewind_to(base + 1)
    got = head.step(7, base + 1)
    want = ohead.step([7], trunk.last_hidden(1), base + 1)[0]
    errs.append(gc.logit_error(got, want))
    print(name, "head logit error / range per step:", ["%.2e" % e for e in errs])
    assert max(errs) <= tol


# the longer prompts go through large passes, which prime the head too (Q8_0: the rotation as a kernel of its own
# under TSV_ROPE_FUSED=0 elsewhere, here the epilogue; routed layers: every expert against the rows that chose it)
@pytest.mark.parametrize("passes", ["64", "prompt"])
@pytest.mark.parametrize("name,n", [("xcd_q4_k", 37), ("xcd_q4_k", 171), ("xcd_q8_0", 171), ("moe_small", 171)])
def test_priming_by_the_prefill_equals_priming_token_by_token(name, n, passes):
    cfg, gpu_a, head_a = _build(name, ctx=200, oracle=False)
    _, gpu_b, head_b = _build(name, ctx=200, oracle=False)
    if passes == "64":
        ffi.check(ffi.lib().tsv_limit_prompt_buffers(gpu_a._h, 0))
    V = cfg["vocab"]
    prompt = np.random.default_rng(6).integers(0, V, n).astype(np.int32)
    la = head_a.prefill_chunk(prompt[:20], 0, next_token=int(prompt[20]))   # two chunks, the first names its next token
    assert head_a.position == 20
    la = head_a.prefill_chunk(prompt[20:], 20)
    assert gc.took(gpu_a, passes if n > 100 else "16")
    for i in range(n):
        lb = gpu_b.produce(int(prompt[i]), i)
        if i + 1 < n:
            head_b.prime(int(prompt[i + 1]), i)
    # (passes of different row counts split their sums differently: equal to rounding, not to the bit)
    assert gc.logit_error(la, lb) <= 5e-4
    assert head_a.position == head_b.position == n - 1
    ka, va = head_a.read_kv(0, n - 1)
    kb, vb = head_b.read_kv(0, n - 1)
    assert np.abs(ka.astype(np.float32) - kb.astype(np.float32)).max() <= 4e-3 * np.abs(kb.astype(np.float32)).max()
    assert np.abs(va.astype(np.float32) - vb.astype(np.float32)).max() <= 4e-3 * np.abs(vb.astype(np.float32)).max()
    assert gc.logit_error(head_a.step(11, n - 1), head_b.step(11, n - 1)) <= 5e-4


# heads whose prompt rows take another route through the kernels: a row of two runs per thread (more than 4096 values), paired
# q / k rows, a value projection in a format of its own; widths that are not whole 256s, projection biases
@pytest.mark.parametrize("name,over", [("xcd_q4_k", dict(hidden=4352, n_q_heads=4, n_kv_heads=2, head_dim=128, ffn=512)),
                                       ("xcd_q4_k", dict(wv=ffi.Q6_K)), ("gptoss_small", {})])
@pytest.mark.parametrize("n,tail", [(65, -1), (81, 5), (172, -1)])
def test_a_prompt_pass_primes_the_head_as_sixteen_rows_at_a_time_do(name, over, n, tail, monkeypatch):
    cfg = dict(synth.CONFIGS[name], max_context=200, **over)
    w = synth.make_weights(cfg, seed=1234)
    hcfg, hw = synth.make_mtp_weights(cfg, w, seed=77)
    if "wv" in over:
        hw["layers"][0]["wv"] = ffi.synth_tensor(over["wv"], 5, 5, 0.02, cfg["n_kv_heads"] * cfg["head_dim"], cfg["hidden"])
    gpu_a = ts.HipVerifier(cfg, w)
    head_a = ts.MtpHead(gpu_a, hcfg, hw)
    monkeypatch.setenv("TSV_WIDE_PREFILL", "0")
    gpu_b = ts.HipVerifier(cfg, w)
    head_b = ts.MtpHead(gpu_b, hcfg, hw)
    prompt = np.random.default_rng(n).integers(0, cfg["vocab"], n).astype(np.int32)
    for head in (head_a, head_b):
        head.prefill_chunk(prompt, 0, next_token=tail)
    assert gc.took(gpu_b, "16") and (n == 65 or gc.took(gpu_a, "prompt"))
    rows = n - (tail < 0)
    assert head_a.position == head_b.position == rows
    # A routed target's rows differ by more where its last expert is a tie to rounding (the two targets' passes sum in another order):
    # 0.4 to 0.7 % of decisions (test_gpu_moe.py), here two a row: six standard deviations above 1.4 % of the rows (6, 7 and 11 of them)
    ties = int(0.014 * rows + 6 * (0.014 * rows) ** 0.5) if cfg.get("n_experts") else 0
    off = np.zeros(rows, bool)
    for a, b in zip(head_a.read_kv(0, rows), head_b.read_kv(0, rows)):
        off |= (np.abs(a.astype(np.float32) - b.astype(np.float32)) > 4e-3 * np.abs(b.astype(np.float32)).max()).any(axis=(1, 2))  # (as above)
    assert off.sum() <= ties, np.flatnonzero(off)
    if tail < 0 and not ties:
        assert gc.logit_error(head_a.step(11, n - 1), head_b.step(11, n - 1)) <= 5e-4


@pytest.mark.parametrize("passes", ["64", "prompt"])
@pytest.mark.parametrize("name,n", [("xcd_q4_k", 64), ("xcd_q4_k", 70), ("xcd_q8_0", 100), ("xcd_q8_0", 128), ("moe_small", 128)])
def test_a_prompt_without_logits_leaves_its_last_rows_for_an_attached_head(name, n, passes, monkeypatch):
    """tsv_prefill on a target with a head keeps the last pass's residual rows (tsv_mtp_open), logits or not: the head
    steps from the last one, as after sixteen-row passes."""
    cfg, gpu_a, head_a = _build(name, ctx=200, oracle=False)
    if passes == "64":
        ffi.check(ffi.lib().tsv_limit_prompt_buffers(gpu_a._h, 0))
    monkeypatch.setenv("TSV_WIDE_PREFILL", "0")
    _, gpu_b, head_b = _build(name, ctx=200, oracle=False)
    prompt = np.random.default_rng(12).integers(0, cfg["vocab"], n).astype(np.int32)
    steps = []
    for gpu, head in ((gpu_a, head_a), (gpu_b, head_b)):
        head.prefill_chunk(prompt, 0)              # the head's cache over [0, n - 1)
        gpu.reset()
        gpu.prefill(prompt, 0, want_logits=False)
        steps.append(head.step(11, n - 1))
    assert gc.logit_error(*steps) <= 5e-4          # the bound of the priming test


@pytest.mark.parametrize("block", [1, 4, 15])
def test_a_block_draft_is_the_chain_of_single_steps(block):
    cfg, gpu, head = _build("small_q4_k", oracle=False)
    V = cfg["vocab"]
    prompt = np.random.default_rng(8).integers(0, V, 18).astype(np.int32)
    n = len(prompt)
    anchor = _amax(head.prefill_chunk(prompt, 0))
    chain, tok = [], anchor
    for d in range(block):
        tok = _amax(head.step(tok, n - 1 + d))
        chain.append(tok)
    head.rewind(n - 1)
    got = head.draft_block(anchor, n, block)
    assert got == chain
    assert head.position == n + block      # the row-only step of the last proposal is in
    # nothing was committed: back to where the round began, and the same block comes out again
    head.rewind(n - 1)
    assert head.draft_block(anchor, n, block) == chain


class _HeadDrafter:
    """The head behind the step-wise drafter methods the reference loop calls."""

    def __init__(self, head):
        self.h = head
        head.rewind(0)

    def prime(self, token, position):
        self.h.prime(token, position)

    def step(self, token, position):
        return self.h.step(token, position)

    def rewind(self, position):
        self.h.rewind(position)


@pytest.mark.parametrize("temperature,kw,block,floor,flags", [
    (0.0, {}, 4, 0, {}),                                     # block drafts, chunked prefill
    (0.0, {}, 8, 2, {}),                                     # adaptive depth
    (0.0, {}, 5, 0, dict(block_drafts=False)),               # the same head step by step
    (0.8, dict(top_p=0.95), 4, 0, {}),                       # sampled rounds: the library's own head chains them on the device
    (0.9, dict(repetition_penalty=1.3, presence_penalty=0.5, top_k=64), 6, 2, {}),   # ... with penalties over the growing history
    (0.8, dict(min_p=0.02), 4, 0, dict(block_drafts=False)), # the same head step by step on device rows
    (0.0, dict(repetition_penalty=1.3), 4, 0, {}),           # the arg-max ignores penalties
])
def test_the_loop_with_the_head_reports_what_the_reference_loop_reports(temperature, kw, block, floor, flags):
    cfg, gpu, head = _build("tiny_q8_0", ctx=200, oracle=False, weak_layers=0.03, follow=16.0)
    V = cfg["vocab"]
    prompt = np.random.default_rng(3).integers(0, V, 19).astype(np.int32)
    seed = 41 if temperature else None
    gcfg, ocfg = ts.shaping(temperature, seed=seed, **kw), ob.shaping(temperature, seed=seed, **kw)
    new = 60
    want = ob.run_speculative(GpuTarget(gpu), _HeadDrafter(head), prompt, ocfg, new, block, V, cfg["max_context"],
                              adaptive_floor=floor)
    got = gpu.run_speculative(prompt, head, gcfg, new, block, adaptive_floor=floor, **flags)
    print({k: (got[k] if k != "tokens" else len(got[k])) for k in KEYS})
    assert {k: got[k] for k in KEYS} == {k: want[k] for k in KEYS}
    assert len(got["tokens"]) == new and got["stop_reason"] == 2
    assert got["kv_position"] == len(prompt) + new - 1 == gpu.position
    assert 0 < got["accepted"] < got["offered"]      # the head proposes what the target picks often, not always
    if temperature == 0.0:
        # greedy speculation is plain decoding
        gpu.reset()
        gpu.prefill(prompt[:-1], 0, want_logits=False)
        tok, plain = int(prompt[-1]), []
        for i in range(new):
            tok = _amax(gpu.produce(tok, len(prompt) - 1 + i))
            plain.append(tok)
        assert got["tokens"] == plain
    # a second run on the same handles starts the head over
    again = gpu.run_speculative(prompt, head, gcfg, new, block, adaptive_floor=floor, **flags)
    assert again["tokens"] == got["tokens"]


def test_refusals_by_name():
    cfg, gpu, head = _build("tiny_q8_0", oracle=False)
    prompt = np.arange(5, 14, dtype=np.int32)
    with pytest.raises(ffi.TsvError, match="holds no row"):
        head.step(3, 0)                                  # nothing has run on the target yet
    head.prefill_chunk(prompt, 0)
    with pytest.raises(ffi.TsvError, match="cache covers"):
        head.step(3, 4)                                  # not where the head's cache ends
    with pytest.raises(ffi.TsvError, match="forward"):
        head.rewind(100)
    with pytest.raises(ffi.TsvError, match="must end where the chunk starts"):
        head.prefill_chunk(prompt, 0)
    with pytest.raises(ffi.TsvError, match="1..15"):
        head.draft_block(3, len(prompt), 16)
    hcfg, hw = synth.make_mtp_weights(cfg, gpu._keep[0], seed=5)
    with pytest.raises(ffi.TsvError, match="already has one"):
        ts.MtpHead(gpu, hcfg, hw)
    with pytest.raises(ffi.TsvError, match="ONE decoder layer"):
        other = ts.HipVerifier(cfg, gpu._keep[0])
        ts.MtpHead(other, dict(hcfg, hidden=cfg["hidden"] * 2), hw)
    # a drafter with neither pair of callbacks
    d = ffi.Drafter()
    ffi.check(ffi.lib().tsv_mtp_drafter(head._h, d))
    d.step = ffi.DRAFT_STEP()
    d.draft_block = ffi.DRAFT_BLOCK()
    import ctypes as C
    g = ffi.Generation()
    g.shaping, g.max_new_tokens, g.block = ts.shaping(0.0), 4, 2
    toks = np.zeros(8, np.int32)
    res = ffi.GenerationResult()
    res.tokens, res.capacity = toks.ctypes.data_as(C.POINTER(C.c_int32)), 8
    rc = ffi.lib().tsv_run_speculative(gpu._h, C.byref(d), prompt.ctypes.data, prompt.size, C.byref(g), C.byref(res))
    assert rc != 0 and "step and prime, or draft_block and prefill_chunk" in ffi.last_error()


def test_a_draw_that_is_refused_ends_the_block_whichever_step_it_is_of():
    """A head whose first step gives every token one score: 1500 penalised candidates between two fp16 values, more than a draw can put in order.
    The steps behind it are sure of their token and need no order, so nothing but the first draw has anything to refuse."""
    V, start, sure, fork = 1600, 1500, 1501, 1502      # tokens below 1500 are the history; `fork` is followed by `start`, that by anything, anything by `sure`
    cfg = dict(synth.CONFIGS["tiny_q8_0"], max_context=1700, vocab=V, weak_layers=0.0)
    w = synth.make_weights(cfg, seed=1)
    hcfg, hw = synth.make_mtp_weights(cfg, w, seed=2, norm_jitter=0.0)
    H = cfg["hidden"]
    e, head = np.zeros((V, H), np.float32), np.zeros((V, H), np.float32)
    e[:, 1], e[start], e[fork] = 1.0, np.eye(H)[0], np.eye(H)[2]
    head[:, 0] = 3.0 / H ** 0.5
    head[sure, 1] = head[start, 2] = 25.0 / H ** 0.5
    w["embed"] = hw["embed"] = ffi.quantize(ffi.BF16, e)
    w["lm_head"] = hw["lm_head"] = ffi.quantize(ffi.BF16, head)
    hw["fc"] = ffi.quantize(ffi.BF16, np.concatenate([np.eye(H), np.zeros((H, H))], axis=1).astype(np.float32))
    gpu = ts.HipVerifier(cfg, w)
    mtp = ts.MtpHead(gpu, hcfg, hw)
    prompt = np.concatenate([np.arange(1500), [fork]]).astype(np.int32)
    refused = 0
    for seed in range(8):
        try:
            gpu.run_speculative(prompt, mtp, ts.shaping(1.0, seed=seed, repetition_penalty=1.1), 6, 4)
        except Exception as err:
            assert "mtp_draft_block" in str(err) and "not built" in str(err), err
            refused += 1
        gpu.reset()
    assert refused >= 4     # the draw falls among the 1500 with 92 %
