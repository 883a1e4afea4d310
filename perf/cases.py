"""The work a user of this library has it do, as measured cases: verify rounds (draft -> forward -> acceptance -> truncation)
over the benchmark configurations, plain decoding, prompts from a short follow-up to thousands of tokens, and the whole
generation loop with the drafter head inside the library -- dense and routed models, every storage type in earnest use,
fp16 and quantized KV rows, greedy and sampled rounds, chains and trees.

A case names a model of turbospark_amd.synth.CONFIGS (or the generic "mid" decoder) with a depth of its own: the layers of a
decoder repeat, so a routed stack of 60 GB is represented by a few of its layers at their real widths, the dense 8B stack is
there in full.  The weights are random and stand for the model file of a user's program: the same ones whatever the seed; the
prompt, the draft and the draws come from the seed.  Two things are arranged so that the values are those of a trained model
rather than of noise: the q and k projections are wide enough for the attention to be peaked, and the output head's row
t + SUCC is the embedding of token t, whose share of the residual stream is that of all layers together -- the model is sure
of its next token, drafts agree with it about as often as published drafters do, and no decision hangs on the last bit of a
logit."""
import functools
import math

import numpy as np
import torch

import turbospark_amd as ts
from turbospark_amd import ffi, synth

SUCC = 17                      # the token the model expects after t is t + SUCC
TREE16 = [-1, 0, 0, 0, 0, 1, 5, 6, 2, 8, 9, 3, 11, 12, 4, 14]   # four children, three chains of depth three, one extra leaf
SIGMA = 0.02
SEED = 20261125                # of the weights

MODELS = dict(synth.CONFIGS)
# a generic decoder between the plumbing case and the 8B shape: 64-wide heads, four q heads to a kv head
MODELS["mid"] = dict(n_layers=16, hidden=2048, n_q_heads=32, n_kv_heads=8, head_dim=64, ffn=8192, vocab=32000, rms_eps=1e-5,
                     rope_theta=500000.0, dtype=ffi.Q4_K)
STORAGE = {"q4_k": ffi.Q4_K, "q4_k_m": ffi.Q4_K, "q5_k_m": ffi.Q5_K, "q8_0": ffi.Q8_0, "bf16": ffi.BF16}

# one case is a dict of: what ("round", "decode", "prompt", "loop"), model, layers, weights (the storage type of a dense
# model's matrices; "own": as the configuration names), context (positions already in the cache), and then
#   round:  rows (1 + proposals), tree, temperature, kv_bits, top_k, top_p, penalty (repetition)
#   decode: tokens (produced one by one)
#   prompt: tokens, kv_bits
#   loop:   tokens (generated), block, temperature; the prompt is `context` tokens, fed by the loop itself
DEFAULTS = dict(weights="own", rows=1, tree=False, temperature=0.0, kv_bits="off", top_k=0, top_p=0.0, penalty=1.0, tokens=0, block=0)


def _case(what, model, layers, context, name=None, **more):
    c = dict(what=what, model=model, layers=layers, context=context)
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: a two-layer decoder, 10 MB of weights; host path and launch count are what it costs
        _case("round", "tiny_q8_0", 2, 256, "tiny_greedy_round", rows=5),
        # the headline step: 8B shape in Q4_K, four proposals, 4096 positions, rejection sampling at 0.8
        _case("round", "llama3_8b_q4_k", 32, 4096, "dense_chain_round", rows=5, temperature=0.8),
        # tree drafts: sixteen rows over a long context, multi-branch rejection
        _case("round", "llama3_8b_q4_k", 16, 16384, "dense_tree_round", rows=16, tree=True, temperature=1.0),
        # the same weights as 8-bit blocks, 4-bit KV rows, the sampling options chat front ends set, an odd context
        _case("round", "llama3_8b_q4_k", 8, 6001, "kv4_shaped_round", weights="q8_0", rows=4, temperature=0.7, kv_bits="4", top_k=40,
              top_p=0.95, penalty=1.1),
        # routed experts, greedy, eight proposals
        _case("round", "qwen3_30b_a3b", 12, 8192, "routed_chain_round", rows=9),
        # gpt-oss layers (bf16 + MXFP4 experts, window / full alternating, sinks) at the long end of the context range
        _case("round", "gptoss_120b", 4, 32768, "gptoss_long_round", rows=9, temperature=1.0),
        # plain decoding without a drafter, the tensor mix of the files most users have
        _case("decode", "llama3_8b_q4_k", 16, 1003, "dense_decode_mix", weights="q4_k_m", tokens=4),
        # a document as prompt
        _case("prompt", "llama3_8b_q4_k", 32, 0, "dense_prompt_2048", tokens=2048),
        # the next turn of a conversation: a few hundred tokens behind a few thousand, not a multiple of anything
        _case("prompt", "llama3_8b_q4_k", 16, 3001, "dense_followup_prompt", weights="q5_k_m", tokens=299),
        # prompts of the routed families
        _case("prompt", "qwen3_30b_a3b", 8, 0, "routed_prompt_1000", tokens=1000),
        _case("prompt", "gptoss_120b", 4, 700, "gptoss_prompt_1500", tokens=1500),
        # everything together: a prompt, then the loop with the library's own drafter head, sampled
        _case("loop", "llama3_8b_q4_k", 8, 400, "dense_generation_loop", tokens=48, block=4, temperature=0.8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["round", "round", "round", "decode", "prompt", "prompt", "prompt", "loop"])
    family = rng.choice(["dense", "dense", "dense", "qwen3_30b_a3b", "gptoss_120b"])
    weights = "own"
    if family == "dense":
        model = rng.choice(["llama3_8b_q4_k", "llama3_8b_q4_k", "mid"])
        weights = rng.choice(["own", "q4_k_m", "q5_k_m", "q8_0", "bf16"])
        layers = rng.randint(2, 12)
    else:
        model, layers = family, rng.randint(2, 6 if family == "qwen3_30b_a3b" else 3)
    kv = rng.choice(["off", "off", "off", "4", "3.5", "2"]) if model != "gptoss_120b" else "off"
    if what == "round":
        tree = family == "dense" and rng.random() < 0.25
        temperature = rng.choice([0.0, 0.7, 1.0])
        more = dict(top_k=40, top_p=0.95) if temperature and not tree and rng.random() < 0.4 else {}
        return _case(what, model, layers, _log(rng, 64, 12000), weights=weights, rows=16 if tree else rng.randint(1, 12), tree=tree,
                     temperature=temperature, kv_bits=kv, **more)
    if what == "decode":
        return _case(what, model, layers, _log(rng, 32, 12000), weights=weights, tokens=rng.randint(1, 8))
    if what == "prompt":
        return _case(what, model, layers, rng.choice([0, _log(rng, 16, 6000)]), weights=weights, tokens=_log(rng, 17, 2500), kv_bits=kv)
    return _case(what, model if family == "dense" else "mid", layers, _log(rng, 50, 1500), weights=weights, tokens=rng.randint(8, 40),
                 block=rng.randint(2, 7), temperature=rng.choice([0.0, 0.8]))


# ---- the model file ------------------------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _pool(dtype, sigma, elems):
    """`elems` N(0, sigma) values as one run of quantized blocks; the matrices of all layers are views into it."""
    cols = 8192
    return ffi.synth_tensor(dtype, SEED, 1 + dtype, sigma, -(-elems // cols), cols)[1].reshape(-1)


@functools.lru_cache(maxsize=8)
def _vocabulary(dtype, sigma, rows, cols):
    return ffi.synth_tensor(dtype, SEED, 77, sigma, rows, cols)[1]


def _config(case):
    cfg = dict(MODELS[case["model"]], n_layers=case["layers"])
    weights = case.get("weights", "own")
    cfg["mix"], cfg["ties"] = weights, case.get("kv_bits", "off") != "off"
    if weights != "own":
        cfg["dtype"] = STORAGE[weights]
    extra = {"round": 32, "decode": case.get("tokens", 0) + 16, "prompt": case.get("tokens", 0) + 32,
             "loop": case.get("tokens", 0) + 32}[case["what"]]
    cfg["max_context"] = case["context"] + extra
    oss = cfg.get("gptoss")
    if oss:
        factor, octx, fast, slow = oss["yarn"]
        cfg["rope_freqs"], cfg["rope_mscale"] = ffi.yarn_frequencies(cfg["head_dim"], cfg["rope_theta"], factor, octx, fast, slow)
        cfg["act_alpha"], cfg["act_limit"] = oss["act_alpha"], oss["act_limit"]
    return cfg


def _vec(rng, n, scale, dtype=ffi.F32, rows=1, offset=0.0):
    v = (offset + rng.standard_normal((rows, n)) * scale).astype(np.float32)
    return (ffi.F32, v.view(np.uint8).reshape(rows, -1), rows, n) if dtype == ffi.F32 else ffi.quantize(dtype, v)


def _higher(l, n):
    """Where a *_K_M file keeps the value and down projections in Q6_K: the first and last eighth and every third layer between."""
    return l < n // 8 or l >= 7 * n // 8 or (l - n // 8) % 3 == 2


def _stream_scale(cfg):
    """The embedding's share of the residual stream: about what all layers add.  Six times that with routed experts, where a
    last expert chosen the other way (about one decision in two hundred lies within the rounding of a tie) moves its row by a
    tenth of what the layers add, and with quantized KV rows, where a coordinate at a code's edge does: a pass is compared by
    its arithmetic, not by its ties."""
    attn = 0.6 * SIGMA * math.sqrt(cfg["n_q_heads"] * cfg["head_dim"])
    ffn = 0.8 * SIGMA * math.sqrt(cfg["ffn"]) / math.sqrt(cfg.get("top_k", 1))
    return math.sqrt(cfg["n_layers"] * (attn * attn + ffn * ffn)) * (6.0 if cfg.get("n_experts") or cfg["ties"] else 1.0)


def _layers(cfg, count, salt0=0):
    H, F, hd = cfg["hidden"], cfg["ffn"], cfg["head_dim"]
    qd, kvd, E = cfg["n_q_heads"] * hd, cfg["n_kv_heads"] * hd, cfg.get("n_experts", 0)
    dt, xd, mix, oss = cfg["dtype"], cfg.get("expert_dtype", cfg["dtype"]), cfg["mix"], cfg.get("gptoss")
    rng = np.random.default_rng(SEED + 3)
    salt = [salt0]

    def t(rows, cols, dtype=None, sigma=SIGMA):
        dtype = dt if dtype is None else dtype
        salt[0] += 1
        need, rb = rows * cols, ffi.row_bytes(dtype, cols)
        pool = _pool(dtype, sigma, max(1 << 26, -(-(need + (1 << 22)) // (1 << 24)) << 24))
        spare = (pool.size - rows * rb) // ffi.row_bytes(dtype, 256)
        at = (salt[0] * 7919 % max(1, spare)) * ffi.row_bytes(dtype, 256)
        return (dtype, pool[at:at + rows * rb].reshape(rows, rb), rows, cols)

    out = []
    for l in range(count):
        high = ffi.Q6_K if mix.endswith("_m") and _higher(l, count) else None
        peak = 0.025 * math.sqrt(4096 / H)      # scores of about 2.5 standard deviations whatever the width
        w = dict(attn_norm=_vec(rng, H, 0.05, offset=1.0), wq=t(qd, H, sigma=peak), wk=t(kvd, H, sigma=peak), wv=t(kvd, H, high),
                 wo=t(H, qd), ffn_norm=_vec(rng, H, 0.05, offset=1.0))
        if cfg.get("qk_norm"):
            w.update(q_norm=_vec(rng, hd, 0.1, offset=1.6), k_norm=_vec(rng, hd, 0.1, offset=1.6))
        if E:
            w.update(n_experts=E, top_k=cfg["top_k"], router=t(E, H, sigma=cfg["router_sigma"]), we_gate=t(E * F, H, xd),
                     we_up=t(E * F, H, xd), we_down=t(E * H, F, xd))
        else:
            w.update(w_gate=t(F, H), w_up=t(F, H), w_down=t(H, F, high))
        if oss:
            w.update(bq=_vec(rng, qd, 0.05, ffi.BF16), bk=_vec(rng, kvd, 0.05, ffi.BF16), bv=_vec(rng, kvd, 0.05, ffi.BF16),
                     bo=_vec(rng, H, 0.05, ffi.BF16), sinks=_vec(rng, cfg["n_q_heads"], 1.0, ffi.BF16),
                     window=oss["window"] if l % 2 == 0 else 0, router_bias=_vec(rng, E, 0.05), be_gate=_vec(rng, F, 0.05, rows=E),
                     be_up=_vec(rng, F, 0.05, rows=E), be_down=_vec(rng, H, 0.05, rows=E))
        out.append(w)
    return out


def _weights(cfg):
    V, H = cfg["vocab"], cfg["hidden"]
    rb = lambda a: a.shape[1]
    head = _vocabulary(ffi.Q6_K if cfg["mix"].endswith("_m") else cfg["dtype"], SIGMA, V + SUCC, H)
    embed = _vocabulary(cfg["dtype"], round(_stream_scale(cfg), 3), V + SUCC, H)
    return dict(embed=(cfg["dtype"], embed[SUCC:], V, H),
                lm_head=(ffi.Q6_K if cfg["mix"].endswith("_m") else cfg["dtype"], head[:V].reshape(V, rb(head)), V, H),
                final_norm=_vec(np.random.default_rng(SEED + 4), H, 0.05, offset=1.0), layers=_layers(cfg, cfg["n_layers"]))


def _head_weights(cfg, weights):
    """A drafter head that has learnt to pass the next token's embedding on: fc near [c I, 0] plus noise."""
    H = cfg["hidden"]
    hcfg = dict(cfg, n_layers=1)
    fc = (np.random.default_rng(SEED + 5).standard_normal((H, 2 * H)) * SIGMA).astype(np.float32)
    fc[:, :H] += 4.0 * np.eye(H, dtype=np.float32)
    layers = _layers(dict(cfg, mix="own"), 1, salt0=500)
    return hcfg, dict(embed=weights["embed"], lm_head=weights["lm_head"], final_norm=weights["final_norm"], layers=layers,
                      fc=ffi.quantize(ffi.Q8_0, fc), norm_embedding=_vec(np.random.default_rng(SEED + 6), H, 0.05, offset=1.0),
                      norm_hidden=_vec(np.random.default_rng(SEED + 7), H, 0.05, offset=1.0))


class _DeviceRows:
    """The logits a pass left on the GPU (rows x vocab fp16), as the library hands out their address; the tensor made from this
    keeps it, and with it the handle that owns the memory."""

    def __init__(self, eng, rows, vocab):
        self.eng = eng
        self.__cuda_array_interface__ = dict(shape=(rows, vocab), typestr="<f2", data=(int(eng.device_logits), False), version=2,
                                             strides=None)


# ---- preparation ------------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    case = dict(DEFAULTS, **case)
    cfg = _config(case)
    weights = _weights(cfg)
    eng = ts.HipVerifier(cfg, weights, kv_bits=ts.producer.parse_kv_bits(case["kv_bits"]))
    rng = np.random.default_rng([seed, 11])
    V, ctx = cfg["vocab"], case["context"]
    state = dict(case=case, eng=eng, vocab=V)
    top = V - SUCC * 64                       # ids from which a chain of successors stays inside the vocabulary
    tokens = rng.integers(0, top, ctx + max(case["tokens"], 1)).astype(np.int32)
    if case["what"] == "loop":
        hcfg, hw = _head_weights(cfg, weights)
        state["head"] = ts.MtpHead(eng, hcfg, hw)
        state["prompt"] = tokens[:ctx]
        state["shaping"] = _shaping(case, seed)
        return state
    if ctx:
        eng.prefill(tokens[:ctx], 0, want_logits=False)
    state["point"], state["base"] = eng.checkpoint(), eng.position
    if case["what"] == "prompt":
        state["tokens"] = tokens[ctx:ctx + case["tokens"]]
    elif case["what"] == "decode":
        state["tokens"] = [int(t) for t in tokens[ctx:ctx + case["tokens"]]]
    else:
        state.update(_draft(case, rng, V, int(rng.integers(0, top))))
        state["shaping"] = _shaping(case, seed)
        state["history"] = np.concatenate([tokens[:ctx][-2000:], [state["feed"][0]]]).astype(np.int32) if case["penalty"] != 1.0 else None
    return state


def _shaping(case, seed):
    if case["temperature"] == 0.0:
        return ts.shaping(0.0)
    return ts.shaping(case["temperature"], seed=seed, top_k=case["top_k"], top_p=case["top_p"] or None, repetition_penalty=case["penalty"])


def _draft(case, rng, V, anchor):
    """The proposals of a round and the drafter's rows they come from: each follows its parent as the model will (seven times
    in ten, one child of a node at most) or is some other token; the row is N(0, 1) noise with its mass on the proposals."""
    m = case["rows"]
    parent = TREE16[:m] if case["tree"] else [i - 1 for i in range(m)]
    feed, right = [anchor], {}
    for s in range(1, m):
        p = parent[s]
        likely = p not in right and rng.random() < (0.4 if case["tree"] and p == 0 else 0.7)
        if likely:
            right[p] = s
        feed.append(feed[p] + SUCC if likely else int(rng.integers(0, V - SUCC * 64)))
    rows = None
    if case["temperature"] > 0.0 and m > 1:
        n = m if case["tree"] else m - 1
        gen = torch.Generator(device="cuda").manual_seed(int(rng.integers(0, 1 << 31)))
        rows = torch.randn((n, V), generator=gen, device="cuda", dtype=torch.float32)
        for s in range(1, m):
            rows[parent[s], feed[s]] = 12.0
        rows = rows.to(torch.float16)
        torch.cuda.synchronize()
    elif case["temperature"] > 0.0:
        rows = torch.zeros((1, V), device="cuda", dtype=torch.float16)
        torch.cuda.synchronize()
    return dict(feed=feed, parent=parent if case["tree"] else None, rows=rows)


# ---- one pass ---------------------------------------------------------------------------------------------------------------

def run(state):
    eng, case = state["eng"], state["case"]
    if case["what"] == "round":
        r = eng.verify_accept(state["feed"], state["base"], state["shaping"], parent=state["parent"],
                              draft_logits=None if state["rows"] is None else state["rows"].data_ptr(), history=state["history"])
        eng.rollback(state["point"])
        logits = torch.as_tensor(_DeviceRows(eng, case["rows"], state["vocab"]), device="cuda")
        path = np.full(case["rows"] + 1, -1, np.int32)
        path[:len(r.path)] = r.path
        return dict(logits=logits, accepted=r.accepted, committed=r.committed, next=r.next, path=path, kv_position=r.kv_position,
                    draw_step=r.draw_step)
    if case["what"] == "decode":
        out = [eng.produce(t, state["base"] + i).view(np.float16) for i, t in enumerate(state["tokens"])]
        eng.rollback(state["point"])
        return out
    if case["what"] == "prompt":
        logits = eng.prefill(state["tokens"], state["base"]).view(np.float16)
        eng.rollback(state["point"])
        return logits
    r = eng.run_speculative(state["prompt"], state["head"], state["shaping"], case["tokens"], case["block"])
    return dict(tokens=np.asarray(r["tokens"], np.int32), stop_reason=r["stop_reason"], rounds=r["rounds"], accepted=r["accepted"],
                draw_step=r["draw_step"], kv_position=r["kv_position"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------------

def _pass_work(cfg, kv_bits, start, rows, heads):
    """Bytes and operations of feeding `rows` rows behind `start` positions in one pass with `heads` rows of logits: every weight
    read once (an expert if any row is expected to choose it), the cache read once and the new rows written, the products of
    the real rows alone."""
    H, F, V, L, hd = cfg["hidden"], cfg["ffn"], cfg["vocab"], cfg["n_layers"], cfg["head_dim"]
    qd, kvd, E, mix, dt = cfg["n_q_heads"] * hd, cfg["n_kv_heads"] * hd, cfg.get("n_experts", 0), cfg["mix"], cfg["dtype"]
    rb = lambda r, c, d: r * ffi.row_bytes(d, c)
    nbytes = flops = 0.0
    for l in range(L):
        high = ffi.Q6_K if mix.endswith("_m") and _higher(l, L) else dt
        nbytes += rb(qd + kvd, H, dt) + rb(kvd, H, high) + rb(H, qd, dt)
        flops += 2.0 * rows * H * (2 * qd + 2 * kvd)
        if E:
            k = cfg["top_k"]
            union = E * (1.0 - (1.0 - k / E) ** rows)
            nbytes += rb(E, H, dt) + union * rb(3 * F, H, cfg.get("expert_dtype", dt))
            flops += 2.0 * rows * H * (E + 3 * F * k)
        else:
            nbytes += rb(2 * F, H, dt) + rb(H, F, high)
            flops += 6.0 * rows * H * F
        window = cfg["gptoss"]["window"] if cfg.get("gptoss") and l % 2 == 0 else 0
        quantized = kv_bits and not window and (L <= 2 or l + 1 < L)
        row = sum(cfg["n_kv_heads"] * (4 + 4 * ((hd * b + 31) // 32)) for b in kv_bits) if quantized else 4 * kvd
        seen = min(window, start) if window else start
        nbytes += row * (seen + rows)
        per_row = min(window, start + rows / 2) if window else start + (rows + 1) / 2
        flops += 4.0 * rows * qd * per_row
    nbytes += rows * ffi.row_bytes(dt, H) + heads * V * 2
    if heads:
        nbytes += rb(V, H, ffi.Q6_K if mix.endswith("_m") else dt)
        flops += 2.0 * heads * H * V
    return nbytes, flops


def work(case):
    case = dict(DEFAULTS, **case)
    cfg, bits, ctx = _config(case), ts.producer.parse_kv_bits(case["kv_bits"]), case["context"]
    if case["what"] == "round":
        parts = [_pass_work(cfg, bits, ctx, case["rows"], case["rows"])]
        if case["temperature"] > 0.0:
            parts.append(((case["rows"] - 1) * cfg["vocab"] * 2.0, 0.0))       # the drafter's rows
    elif case["what"] == "decode":
        parts = [_pass_work(cfg, bits, ctx + i, 1, 1) for i in range(case["tokens"])]
    elif case["what"] == "prompt":
        parts = [_pass_work(cfg, bits, ctx, case["tokens"], 1)]
    else:
        # the prompt once through target and head, then rounds that each yield block + 1 tokens, block head steps before each
        head = dict(cfg, n_layers=1, mix="own")
        parts = [_pass_work(cfg, bits, 0, ctx, 1), _pass_work(head, bits, 0, ctx, 0)]
        for i in range(0, case["tokens"] - 1, case["block"] + 1):
            parts.append(_pass_work(cfg, bits, ctx + i, case["block"] + 1, case["block"] + 1))
            parts += [_pass_work(head, bits, ctx + i, 1, 1)] * case["block"]
    return dict(bytes=sum(p[0] for p in parts), flops=sum(p[1] for p in parts))


def tolerance(case):
    # The same passes with their sums in another order (16-row prompt passes, the other matrix-instruction forms, the rotation
    # in a kernel of its own), all listed and sixty drawn cases: 4e-4 to 7e-4 of the logits' norm and at most 3.4e-3 of a logit
    # with dense layers; routed ones 2e-4 to 4e-4, more where a tie between experts falls the other way; quantized KV rows
    # 2e-3 to 7e-3, as codes flip.  The loop's tokens and counts are whole numbers.
    case = dict(DEFAULTS, **case)
    if case["what"] == "loop":
        return "exact"
    if case["kv_bits"] != "off":
        return dict(rel=0.025, max=0.2)
    if MODELS[case["model"]].get("n_experts"):
        return dict(rel=0.006, max=0.1)
    return dict(rel=0.003, max=0.015)
