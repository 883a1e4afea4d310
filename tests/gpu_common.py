"""Shared helpers of the GPU parity tests: model construction on both sides, tolerances."""
import ctypes as C
import os

import numpy as np

import turbospark_amd as ts
from turbospark_amd import ffi, synth
from oracle import binding as ob


def f16(bits):
    return np.asarray(bits, np.uint16).view(np.float16).astype(np.float32)


def build_pair(name, max_context, seed=1234, threads=8, **over):
    cfg = dict(synth.CONFIGS[name])
    cfg.update(over)
    cfg["max_context"] = max_context
    weights = synth.make_weights(cfg, seed=seed)
    gpu = ts.HipVerifier(cfg, weights)
    cpu = ob.Model(cfg, weights, round_kv_f16=True, threads=threads)
    return cfg, weights, gpu, cpu


def logit_error(got_bits, want_bits):
    """max |got - want| relative to the reference row's logit range (the north-star metric)."""
    g, w = f16(got_bits), f16(want_bits)
    rng = (w.max(axis=-1) - w.min(axis=-1)).max()
    return float(np.abs(g - w).max() / rng)


def prompt_buffers(eng):
    """(rows of the longest prompt pass, bytes held, prompt passes so far, 64-row passes so far)"""
    rows, held, passes = C.c_int32(), C.c_int64(), (C.c_int64 * 2)()
    ffi.check(ffi.lib().tsv_prompt_buffers(eng._h, C.byref(rows), C.byref(held), passes))
    return rows.value, held.value, passes[0], passes[1]


def engine(cfg, weights, passes, **kw):
    """A handle whose prompts go in "prompt" passes (of up to 2048 rows), in passes of "64" rows, or of "16"."""
    os.environ["TSV_WIDE_PREFILL"] = "0" if passes == "16" else "1"
    try:
        eng = ts.HipVerifier(cfg, weights, **kw)
    finally:
        del os.environ["TSV_WIDE_PREFILL"]
    if passes == "64":
        ffi.check(ffi.lib().tsv_limit_prompt_buffers(eng._h, 0))
    return eng


def took(eng, passes):
    """Whether the handle's prompts so far went that way: prompt passes and no 64-row ones, the other way round, or neither."""
    _, _, prompt, blocks = prompt_buffers(eng)
    return (prompt > 0, blocks > 0) == (passes == "prompt", passes == "64")


TOL = {ffi.Q8_0: 2e-3, ffi.Q4_K: 1e-2, ffi.Q5_K: 1e-2}
