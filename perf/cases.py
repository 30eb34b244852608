"""The calls whose speed is measured, through the framework's public entry points.

A case is one call (or one session of step-wise calls) that a program which
holds a loaded model makes on new data: token ids or coded chunks in host
memory (device memory for the allocation-free entry point) in, coded bytes,
token ids or coder intervals out.  Loading the model is not part of a pass: a
program keeps it (`_model`).

Models: the shipped `v001_eng.czm` on tokenized text, and the two random-init
shapes of `czip_amd.synth.MODEL_SHAPES` on Zipf(1.1) ids: d512 / 8 layers, and
d768 / 12 layers with a vocabulary of 8192 (GQA).

Every output is bytes or whole numbers defined bit for bit, so every tolerance
is "exact".
"""
from __future__ import annotations

import ctypes
import functools
import math
import os
import sys
import tempfile

import numpy as np
import torch

_PKG = os.path.abspath("compress-zip_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import czip_amd  # noqa: E402
from czip_amd import synth  # noqa: E402

SHIPPED = dict(d=384, n_layers=1, n_heads=6, n_kv=1, d_ff=1024, vocab=1024, ctx=1024)
# drawn sizes: the most tokens of one call per model, those of the largest listed cases
COMPRESS_MAX = {"v001": 19_650_003, "d512_l8": 1_000_003, "d768_l12": 200_001}
INTERVAL_ROWS_MAX = 18_944  # rows that fit the allocation-free entry point's buffer


def _shape(model):
    return SHIPPED if model == "v001" else synth.MODEL_SHAPES[model]


def listed():
    return [
        # a short message compressed at the CLI's default level (64-token chunks): latency of one call
        dict(name="compress_message", op="compress", model="v001", kv="rust", tokens=173, chunk=64),
        # the 32 KiB file of the parity configuration, level 1: 418 chunks of 64
        dict(name="compress_32KiB_L1", op="compress", model="v001", kv="rust", tokens=26_709, chunk=64),
        # 24 MiB of text at level 4: the headline workload's model, level and data
        dict(name="compress_24MiB_L4", op="compress", model="v001", kv="rust", tokens=19_650_003, chunk=512),
        # a one-page note at level 4: two streams, 512 dependent steps
        dict(name="decompress_page_L4", op="decompress", model="v001", kv="rust", tokens=850, chunk=512),
        # the 75 KB of the published article sample at level 4: 115 streams
        dict(name="decompress_75KB_L4", op="decompress", model="v001", kv="rust", tokens=58_711, chunk=512),
        # 24 MiB of text at level 4: 38 thousand streams
        dict(name="decompress_24MiB_L4", op="decompress", model="v001", kv="rust", tokens=19_650_003, chunk=512),
        # coder intervals of 37 ragged chunks for a caller with its own encoder, device buffers, no allocation
        dict(name="intervals_device_37x512", op="intervals", model="v001", kv="rust", streams=37, chunk=512, device=True),
        # the d512 model at level 5 (1024-token chunks), a million ids
        dict(name="compress_d512_1M_L5", op="compress", model="d512_l8", kv="rust", tokens=1_000_003, chunk=1024),
        # its decoding configuration: 4096 streams of 512 tokens (the last one shorter)
        dict(name="decompress_d512_4096x512", op="decompress", model="d512_l8", kv="rust", tokens=2_096_999, chunk=512),
        # the d768 GQA model at its 4096-token context
        dict(name="compress_d768_200K_ctx4096", op="compress", model="d768_l12", kv="gqa", tokens=200_001, chunk=4096),
        # the d768 GQA model on a file of an ordinary size: 59 streams of 256
        dict(name="decompress_d768_15K", op="decompress", model="d768_l12", kv="gqa", tokens=15_001, chunk=256),
        # step-wise decoding for callers that keep their own decoder: 48 ragged streams, one call a token
        dict(name="decode_steps_d768_48x64", op="steps", model="d768_l12", kv="gqa", streams=48, chunk=64, tables=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["compress", "decompress", "compress", "decompress", "intervals", "steps"])
    model = rng.choice(["v001", "v001", "d512_l8", "d768_l12"])
    kv = {"v001": "rust", "d512_l8": rng.choice(["rust", "gqa"]), "d768_l12": "gqa"}[model]
    case = dict(op=op, model=model, kv=kv)
    levels = [64, 128, 256, 512, 1024]
    if op == "compress":
        case["chunk"] = rng.choice(levels + ([4096] if model == "d768_l12" else []))
        case["tokens"] = _log_int(rng, 100, COMPRESS_MAX[model] * 512 // max(512, case["chunk"]))
    elif op == "decompress":
        if model == "v001":
            case["chunk"] = rng.choice(levels)
            case["tokens"] = _log_int(rng, 100, COMPRESS_MAX[model] * 512 // max(512, case["chunk"]) // 2)
        elif model == "d512_l8":
            case["chunk"] = rng.choice([64, 128, 256, 512])
            case["tokens"] = _log_int(rng, 100, 4096 * case["chunk"])
        else:
            case["chunk"] = rng.choice([64, 128, 256])
            case["tokens"] = _log_int(rng, 100, 128 * case["chunk"])
    elif op == "intervals":
        case.update(model="v001", kv="rust", chunk=rng.randint(1, 1024), device=rng.random() < 0.5)
        case["streams"] = _log_int(rng, 1, max(2, INTERVAL_ROWS_MAX // case["chunk"]))
        if case["streams"] * case["chunk"] > INTERVAL_ROWS_MAX:
            case["streams"] = 1
    else:
        case.update(streams=_log_int(rng, 1, 512), chunk=rng.randint(8, 96), tables=rng.random() < 0.25)
        if case["tables"]:  # [S, V] tables every step: at most 64 MiB in all
            case["streams"] = max(1, min(case["streams"], (16 << 20) // (case["chunk"] * _shape(model)["vocab"])))
    return case


@functools.lru_cache(maxsize=None)
def _model(name, kv):
    mode = czip_amd.KV_GQA if kv == "gqa" else czip_amd.KV_RUST_COMPAT
    if name == "v001":
        return czip_amd.Model(czip_amd.ModelWeights(os.path.join("models", "v001_eng.czm"), mode), device=0)
    with tempfile.TemporaryDirectory(prefix="czip_cases_") as tmp:
        path = os.path.join(tmp, name + ".czm")
        synth.write_random_model(path, seed=2024, **synth.MODEL_SHAPES[name])
        return czip_amd.Model(czip_amd.ModelWeights(path, mode), device=0)


@functools.lru_cache(maxsize=None)
def _tokenizer():
    return czip_amd.Tokenizer(_model("v001", "rust").weights)


def _ids(model, n, seed):
    """n token ids: tokenized text for the shipped model, Zipf ids for the others."""
    if model != "v001":
        return synth.zipf_ids(n, _shape(model)["vocab"], seed=seed)
    have = n + n // 3 + 64
    while True:  # about 1.28 bytes a token
        ids = _tokenizer().encode(synth.synthetic_text(have, seed=seed), threads=8)
        if ids.size >= n:
            return ids[:n].copy()
        have += have // 4


def _counts(case):
    n, t = case["tokens"], case["chunk"]
    return [min(t, n - i) for i in range(0, n, t)]


def _lens(case, seed):
    """Ragged stream lengths in [1, chunk], the first one full."""
    rng = np.random.default_rng([seed, 1])
    lens = rng.integers(1, case["chunk"] + 1, case["streams"]).astype(np.int32)
    lens[rng.random(lens.size) < 0.5] = case["chunk"]
    lens[0] = case["chunk"]
    return lens


def prepare(case, seed):
    m = _model(case["model"], case["kv"])
    st = dict(op=case["op"], model=m, chunk=case["chunk"])
    if case["op"] == "compress":
        st["ids"] = _ids(case["model"], case["tokens"], seed)
        nchunks = len(_counts(case))
        st["out"] = np.zeros(nchunks * czip_amd.lib().czip_chunk_slot_bytes(case["chunk"]), np.uint8)
        st["offs"] = np.zeros(nchunks + 1, np.int64)
    elif case["op"] == "decompress":
        st["chunks"] = m.compress_chunks(_ids(case["model"], case["tokens"], seed), case["chunk"])
        st["ntoks"] = np.array(_counts(case), np.int32)
    elif case["op"] == "intervals":
        s, t = case["streams"], case["chunk"]
        st["ids"] = _ids(case["model"], s * t, seed).reshape(s, t)
        st["lens"] = _lens(case, seed)
        st["device"] = case["device"]
        if case["device"]:
            st["d_ids"] = torch.from_numpy(st["ids"].view(np.int32)).cuda()
            st["d_lens"] = torch.from_numpy(st["lens"]).cuda()
            st["d_out"] = torch.zeros((s, t, 2), dtype=torch.int32, device="cuda")
    else:
        s, t = case["streams"], case["chunk"]
        rng = np.random.default_rng([seed, 2])
        ids = _ids(case["model"], s * t, seed).reshape(t, s)
        pos = np.arange(t, dtype=np.int32)[:, None]
        st["streams"] = s
        st["pos"] = np.where(pos < _lens(case, seed)[None, :], pos, -1).astype(np.int32)
        st["tok_in"] = np.concatenate([np.full((1, s), czip_amd.BOS, np.uint32), ids[:-1]])
        st["values"] = None if case["tables"] else rng.integers(0, m.target_total, (t, s)).astype(np.uint32)
    return st


def run(state):
    m = state["model"]
    if state["op"] == "compress":
        job = m.compress_plan(state["ids"], state["chunk"])
        try:
            job.run()
            out, offs = state["out"], state["offs"]
            m._check(czip_amd.lib().czip_compress_fetch_packed(job.h, out.ctypes.data, out.size, offs.ctypes.data))
        finally:
            job.free()
        return [out, offs]
    if state["op"] == "decompress":
        return m.decompress_chunks(state["chunks"], state["ntoks"])
    if state["op"] == "intervals":
        if not state["device"]:
            return m.prefill_cdf(state["ids"], state["lens"])
        s, t = state["ids"].shape
        m._check(czip_amd.lib().czip_prefill_cdf_noalloc(
            m._ctx, ctypes.c_void_p(state["d_ids"].data_ptr()), ctypes.c_void_p(state["d_lens"].data_ptr()), s, t,
            ctypes.c_void_p(state["d_out"].data_ptr())))
        return state["d_out"]
    out = []
    m.decode_begin(state["streams"], state["chunk"])
    try:
        for p in range(state["chunk"]):
            values = None if state["values"] is None else state["values"][p]
            out.append(m.decode_step(state["tok_in"][p], state["pos"][p], values))
    finally:
        m.decode_end()
    return np.stack(out)


def work(case):
    """int8 multiply-adds (two operations each) of the model's products (layer
    0's Q/K/V projection depends on the token alone and can be a table) and of
    the causal attention; bytes: the weights once, inputs and outputs once, and
    for decoding the cached keys and values a step has to read, where the
    caches are larger than the chip's own caches hold (256 MB)."""
    sh = _shape(case["model"])
    d, L, F, V = sh["d"], sh["n_layers"], sh["d_ff"], sh["vocab"]
    kvh = sh["n_kv"] if case["kv"] == "gqa" else 1
    qkv = (d + 128 * kvh) * d
    weights = V * d * 2 + L * (qkv + d * d + 3 * F * d)
    if case["op"] in ("compress", "decompress"):
        full, rest = divmod(case["tokens"], case["chunk"])
        n = case["tokens"]
        pairs = full * case["chunk"] * (case["chunk"] + 1) // 2 + rest * (rest + 1) // 2
        streams = full + (rest > 0)
        moved = 5 * n  # 4-byte ids on one side, about one coded byte a token on the other
    else:
        # half of the streams are full, the others uniform: three quarters of the rows are live
        n = case["streams"] * case["chunk"] * 3 // 4
        pairs = case["streams"] * case["chunk"] * (case["chunk"] + 1) // 3
        streams = case["streams"]
        moved = n * (4 * V + 4 if case.get("tables") else 20)
    flops = 2 * n * ((L - 1) * qkv + L * (d * d + 3 * F * d) + V * d) + 4 * L * d * pairs
    if case["op"] in ("decompress", "steps") and L * streams * case["chunk"] * kvh * 128 > 256e6:
        moved += L * kvh * 128 * pairs
    return {"bytes": int(weights + moved), "flops": int(flops)}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """What a decompression returns is what was coded.  The other outputs are
    defined by an integer chain with its own rounding at every step, which has
    no counterpart in 64-bit arithmetic; they are compared bit for bit."""
    if case["op"] != "decompress":
        return None
    return _ids(case["model"], case["tokens"], seed)
