"""The work this framework is used for, as cases a timing harness can run.

Every case builds a `Model` (one tensor-parallel shard of a stack of layers, assembled as launch vectors by the C++ runtime)
and takes one step through its public entry points: a prefill (`run`), a prefill in chunks over the KV cache (`run_chunked`),
a decode step over equally long sequences (`run_decode`) or over sequences of different lengths in scattered cache slots
(`run_decode_seqs`), or a queue of requests drained by the `Scheduler`.  Activations and cached keys / values are N(0, 1),
weights N(0, 0.02), as in the repository's tests and benchmark.
"""
import ctypes
import importlib
import math

import torch

capi = importlib.import_module("24ppopp-liger_amd.capi")
host = importlib.import_module("24ppopp-liger_amd.host")

# Options a case may leave out, at the values of Model()'s own arguments.
DEFAULTS = {"dtype": "f16", "layers": 1, "shards": 1, "pre_ln": False, "causal": False, "fused": False, "layout": 0,
            "geglu": False, "packed": False, "cache_len": 0}


def listed():
    glm = {"heads": 96, "d": 128, "shards": 2, "ffn": 32768, "causal": True}        # one GPU's TP=2 shard, GLM-130B-shaped
    fast = dict(glm, fused=True, layout=2, packed=True)                             # as the benchmark assembles it
    return [
        # The smallest call in use: one BERT-style layer, fp32, pre-LayerNorm, 64 tokens.  Launches and host time.
        {"name": "small_layer_fp32", "kind": "prefill", "dtype": "f32", "heads": 4, "d": 64, "ffn": 1024, "pre_ln": True, "batch": 2, "seq": 32},
        # An ordinary encoder in fp32 with every option at its default: two layers, hidden 1024, 800 tokens of odd shape.
        {"name": "encoder_fp32", "kind": "prefill", "dtype": "f32", "heads": 16, "d": 64, "ffn": 4096, "layers": 2, "batch": 4, "seq": 200},
        # The load of the published serving experiment: 128 heads of 96, four layers, two short sequences (16 to 115 tokens),
        # assembled as the command-line driver does.
        {"name": "served_short", "kind": "prefill", "heads": 128, "d": 96, "shards": 2, "ffn": 49152, "layers": 4, "fused": True, "layout": 1,
         "batch": 2, "seq": 53},
        # The launch vector in the reference's shape (separate bias, softmax and transpose kernels), weights [in, out], at the
        # shard's full width and a ragged length: what a user gets who changes nothing but the library.
        {"name": "reference_vector", "kind": "prefill", **glm, "batch": 2, "seq": 333},
        # The headline prefill: 8 sequences of 512 tokens, causal.
        {"name": "prefill_batch", "kind": "prefill", **fast, "batch": 8, "seq": 512},
        # One arriving prompt of a serving trace, K and V written into its cache slot, two layers.
        {"name": "prefill_prompt", "kind": "prefill", **fast, "layers": 2, "cache_len": 1088, "batch": 1, "seq": 384},
        # A long prompt taken in chunks over its cache slot, gated FFN as in the GLM family.
        {"name": "prefill_chunked", "kind": "chunked", **fast, "geglu": True, "cache_len": 1088, "seq": 1000, "chunk": 256},
        # The headline decode step: 32 sequences with 1024 cached positions.
        {"name": "decode_batch", "kind": "decode", **fast, "cache_len": 1088, "batch": 32, "past": 1024},
        # A decode step of one sequence alone (latency), weights [out, in], separate projections, two layers.
        {"name": "decode_single", "kind": "decode", **glm, "fused": True, "layout": 1, "layers": 2, "cache_len": 1088, "batch": 1, "past": 777},
        # A large decode batch: more token rows than the few-row kernels take.
        {"name": "decode_wide", "kind": "decode", **fast, "cache_len": 576, "batch": 80, "past": 500},
        # Decode steps of different requests as one step, sequences of different lengths, a whole (unsharded) layer of hidden
        # 4096 with a gated FFN and weights [in, out].
        {"name": "decode_ragged", "kind": "decode_seqs", "heads": 32, "d": 128, "ffn": 16384, "causal": True, "fused": True, "geglu": True,
         "cache_len": 1088, "batch": 11, "past": 1000},
        # The scheduler draining a mixed queue: prompts of different lengths, each followed by decode steps that requests share.
        # With residual connections, as every layer has that is meant to be iterated: without them one step's rounding grows
        # two and a half times with every step that follows (random weights), and no two summation orders can be compared.
        {"name": "queue_mixed", "kind": "queue", **fast, "pre_ln": True, "cache_len": 576, "requests": 6, "seq": 500, "steps": 6},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_once(rng):
    kind = rng.choices(["f32", "vector", "prefill", "chunked", "decode", "decode_seqs", "queue"], [3, 3, 5, 2, 5, 2, 1])[0]
    if kind == "f32":
        heads, d = rng.choice([(4, 64), (8, 64), (12, 64), (16, 64), (8, 96), (8, 128)])
        return {"kind": "prefill", "dtype": "f32", "heads": heads, "d": d, "ffn": 4 * heads * d, "layers": rng.choice([1, 2]),
                "pre_ln": rng.random() < 0.5, "causal": rng.random() < 0.5, "layout": rng.choice([0, 1]),
                "batch": _log_int(rng, 1, 8), "seq": _log_int(rng, 8, 512)}
    heads, d, shards, ffn = rng.choice([(8, 128, 1, 4096), (16, 128, 1, 8192), (32, 128, 1, 16384), (96, 128, 2, 32768), (128, 96, 2, 49152)])
    c = {"heads": heads, "d": d, "shards": shards, "ffn": ffn, "layers": rng.choice([1, 1, 2]), "causal": True,
         "layout": rng.choice([0, 1, 2, 2]), "geglu": rng.random() < 0.3, "packed": rng.random() < 0.5, "pre_ln": rng.random() < 0.3}
    if kind == "vector":
        c.update(kind="prefill", causal=rng.random() < 0.7, batch=_log_int(rng, 1, 4), seq=_log_int(rng, 16, 512))
    elif kind == "prefill":
        c.update(kind="prefill", fused=True, batch=_log_int(rng, 1, 8), seq=_log_int(rng, 16, 1024))
        if rng.random() < 0.5:
            c["cache_len"] = 1088
    elif kind == "chunked":
        c.update(kind="chunked", fused=True, cache_len=1088, seq=_log_int(rng, 300, 1088), chunk=rng.choice([128, 200, 256, 384, 512]))
    elif kind == "decode":
        c.update(kind="decode", fused=True, cache_len=1088, batch=_log_int(rng, 1, 128), past=_log_int(rng, 16, 1087))
    elif kind == "decode_seqs":
        c.update(kind="decode_seqs", fused=True, layers=1, cache_len=1088, batch=_log_int(rng, 2, 24), past=_log_int(rng, 64, 1087))
    else:
        c.update(kind="queue", fused=True, pre_ln=True, layers=1, cache_len=576, requests=rng.randint(3, 8), seq=rng.randint(100, 512), steps=rng.randint(2, 8))
    return c


def _cost(case):
    """A rough time of a pass, to keep drawn cases within the largest listed one."""
    w = work(case)
    return w["flops"] / (1e14 if case.get("dtype") == "f32" else 1e15) + w["bytes"] / 5e12


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw_once(rng)
        if _cost(c) <= most:
            return c


def _full(case):
    return {**DEFAULTS, **case}


def _lengths(c):
    """Cached positions of the sequences of a ragged decode step: from a quarter of `past` up to it, in no order."""
    n, hi = c["batch"], c["past"]
    lo = max(1, hi // 4)
    return [lo + (hi - lo) * ((7 * i + 3) % n) // max(1, n - 1) for i in range(n)]


def _prompts(c):
    """Prompt lengths of a queue: from a fifth of `seq` up to it."""
    n, hi = c["requests"], c["seq"]
    lo = max(16, hi // 5)
    return [lo + (hi - lo) * ((5 * i + 2) % n) // max(1, n - 1) for i in range(n)]


class _Memory:
    """Device memory of the framework (a KV cache, a request's buffers) shown to torch.  torch keeps this object for as long as
    a tensor uses the memory, and it keeps the model or scheduler that frees the memory when it goes."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f2", "data": (ptr, False), "version": 2, "strides": None}


def _view(owner, ptr, *shape):
    return torch.as_tensor(_Memory(owner, ptr, shape), device="cuda")


_stream = None


def _serving_stream():
    """The stream that a serving process launches its steps on, one after the other."""
    global _stream
    if _stream is None:
        p = ctypes.c_void_p()
        capi.check(capi.lib.lg_stream_create(ctypes.byref(p)), "lg_stream_create")
        _stream = p.value
    return _stream


def _model(c, max_batch, max_seq, seed):
    return host.Model(capi.F16 if c["dtype"] == "f16" else capi.F32, max_batch, max_seq, c["heads"], c["d"], layer_num=c["layers"],
                      world_size=c["shards"], ffn_inner=c["ffn"], norm_mode=host.PRE_LN_RESID if c["pre_ln"] else host.POST_NORESID,
                      causal=c["causal"], fused=c["fused"], max_cache_len=c["cache_len"], weight_layout=c["layout"], seed=seed,
                      ffn_act=host.FFN_GEGLU if c["geglu"] else host.FFN_GELU, packed_qkv=c["packed"])


def _caches(m, c, slots):
    """[(k, v)] of every layer, [slots, local heads, cache_len, d]."""
    shape = (slots, c["heads"] // c["shards"], c["cache_len"], c["d"])
    return [tuple(_view(m, p, *shape) for p in m.kv_cache(layer)) for layer in range(c["layers"])]


def prepare(case, seed):
    c = _full(case)
    kind, seed = c["kind"], int(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    hidden = c["heads"] * c["d"]
    dtype = torch.float16 if c["dtype"] == "f16" else torch.float32
    s = {"case": c, "stream": _serving_stream()}

    if kind == "queue":
        n = c["requests"]
        top = (c["seq"] + 63) // 64 * 64
        m = s["model"] = _model(c, n + 1, top, seed)
        sched = s["scheduler"] = host.Scheduler(m, policy=host.POLICY_RESOURCE, axis=host.SPLIT_TOKEN_ROWS, seq_bucket=64, pool_count=n, ctx_batch=1)
        sched.profile(1, 64, top, 64, 2)
        for past in range(64, top + 65, 64):
            for rows in (1, 2, 4):
                sched.profile_decode(rows, min(past, c["cache_len"] - 1), 2)
        sched.set_merge_minor(True)
        sched.enable_batch_decode(True, 2)
        s["requests"] = _prompts(c)
        s["outputs"] = []
        k, v = _caches(m, c, n + 1)[0]
        for i, seq in enumerate(s["requests"]):
            x, y = sched.ctx_ptrs(i)
            _view(sched, x, seq, hidden).copy_(torch.randn(seq, hidden, generator=gen, device="cuda", dtype=dtype))
            last = sched.ctx_decode_ptrs(i)[c["steps"] % 2]
            filled = seq + c["steps"]
            s["outputs"] += [_view(sched, y, seq, hidden), _view(sched, last, 1, hidden), k[i, :, :filled], v[i, :, :filled]]
        torch.cuda.synchronize()
        return s

    batch, rows = {"prefill": (c.get("batch"), c.get("seq")), "chunked": (1, c.get("seq")),
                   "decode": (c.get("batch"), 1), "decode_seqs": (c.get("batch"), 1)}[kind]
    slots = batch if kind != "decode_seqs" else batch + 5
    m = s["model"] = _model(c, slots, rows, seed)
    s["x"] = torch.randn(batch * rows, hidden, generator=gen, device="cuda", dtype=dtype)
    s["y"] = torch.empty_like(s["x"])
    s["outputs"] = [s["y"]]
    if c["cache_len"]:
        caches = _caches(m, c, slots)
        for k, v in caches:
            if kind in ("decode", "decode_seqs"):
                k.normal_(generator=gen)
                v.normal_(generator=gen)
            if kind == "decode":
                s["outputs"] += [k[:, :, c["past"]], v[:, :, c["past"]]]
            elif kind == "decode_seqs":
                s["pasts"] = _lengths(c)
                s["slots"] = [(i * 3 + 1) % slots if slots % 3 else i for i in range(batch)]
                for slot, past in zip(s["slots"], s["pasts"]):
                    s["outputs"] += [k[slot, :, past], v[slot, :, past]]
            else:
                s["outputs"] += [k[:, :, :c["seq"]], v[:, :, :c["seq"]]]
    torch.cuda.synchronize()
    return s


def run(s):
    c, m = s["case"], s["model"]
    kind = c["kind"]
    if kind == "prefill":
        m.run(s["x"].data_ptr(), s["y"].data_ptr(), c["batch"], c["seq"], None, s["stream"], 0 if c["cache_len"] else -1)
    elif kind == "chunked":
        m.run_chunked(s["x"].data_ptr(), s["y"].data_ptr(), c["seq"], c["chunk"], 0, None, s["stream"])
    elif kind == "decode":
        m.run_decode(s["x"].data_ptr(), s["y"].data_ptr(), c["batch"], c["past"], 0, None, s["stream"])
    elif kind == "decode_seqs":
        m.run_decode_seqs(s["x"].data_ptr(), s["y"].data_ptr(), s["slots"], s["pasts"], None, s["stream"])
    else:
        for seq in s["requests"]:
            s["scheduler"].serve(1, seq, c["steps"])
        s["scheduler"].run_queued(host.MODE_LIGER)
    return s["outputs"]


def work(case):
    """Weights, inputs, cached keys and values read once, outputs and new keys and values written once; the matrix products of
    the layer and of the attention (half of the scores where the mask is causal)."""
    c = _full(case)
    es = 2 if c["dtype"] == "f16" else 4
    hidden, hl, ffn = c["heads"] * c["d"], c["heads"] * c["d"] // c["shards"], c["ffn"] // c["shards"]
    weights = c["layers"] * (4 * hidden * hl + (3 if c["geglu"] else 2) * hidden * ffn)

    def step(batch, seq, past, reads_cache):
        tokens = batch * seq
        pairs = tokens * (past + ((seq + 1) / 2 if c["causal"] and seq > 1 else seq))
        moved = 2 * tokens * hidden + (2 * c["layers"] * tokens * hl if c["cache_len"] else 0) + (2 * c["layers"] * batch * past * hl if reads_cache else 0)
        return moved * es, 2.0 * tokens * weights + 4.0 * c["layers"] * pairs * hl

    kind = c["kind"]
    if kind == "prefill":
        parts = [step(c["batch"], c["seq"], 0, False)]
    elif kind == "chunked":
        parts = [step(1, c["seq"], 0, False)]
    elif kind == "decode":
        parts = [step(c["batch"], 1, c["past"], True)]
    elif kind == "decode_seqs":
        parts = [step(1, 1, past, True) for past in _lengths(c)]
    else:
        parts = [step(1, seq, 0, False) for seq in _prompts(c)]
        parts += [step(1, 1, seq + t, True) for seq in _prompts(c) for t in range(c["steps"])]
    # the decode steps of a queue may share a pass over the weights: one pass for each step index, one for the prompts together
    passes = 1 + c["steps"] if kind == "queue" else 1
    return {"bytes": float(passes * weights * es + sum(p[0] for p in parts)), "flops": float(sum(p[1] for p in parts))}


def tolerance(case):
    """About four times what one implementation showed against the same layers computed by torch with fp64 sums and the same
    roundings between the kernels: fp32 1.6e-6 (largest element 8.4e-6 after two layers), fp16 6e-4 (one layer, fused) to 2.2e-3
    (four layers), largest element 1.2e-2."""
    if _full(case)["dtype"] == "f32":
        return {"rel": 6e-6, "max": 4e-5}
    return {"rel": 8e-3, "max": 5e-2}
