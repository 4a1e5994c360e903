"""The workloads this package is timed on, each one pass through its public entry points.

Every case goes in through the layer-level caller, `FlashAttention.compute_attention`, as a model does:
the dispatch picks the kernel, the kernel runs, and for a training case autograd hands back the
gradients.  A paged decode step first writes the step's new keys and values into the page pool
(`paged_extend_step`), as a serving loop does.

  listed()         the cases that are timed
  draw(rng)        one more case of the same ranges
  prepare(c, seed) what the caller holds before the call: projections, cache or pool, biases, the layer
  run(state)       one pass; returns all it computes
  work(c)          bytes and operations the pass cannot do without
  tolerance(c)     how far another correct implementation of the same precision may be off

A case is one of three kinds: "decode" (one query token per sequence over a contiguous cache or a page
pool), "chunk" (some query rows per sequence, each chunk at its own offset into a contiguous cache) and
"self" (prefill or training over whole sequences).
"""

import random

import numpy as np
import torch

from axlearn_amd import attention_bias as ab
from axlearn_amd.flash_attention.layer import FlashAttention
from axlearn_amd.kv_cache import KVCache, PagedKVCache, paged_extend_step

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
MAX_DOCS = 6          # documents packed into one row of a packed training batch


def _decode(name=None, **kw):
    c = dict(kind="decode", batch=1, capacity=1024, shortest=1024, q_heads=8, kv_heads=8, head_dim=128, page=0,
             window=-1, dtype="bf16")
    return _case(c, name, kw)


def _chunk(name=None, **kw):
    c = dict(kind="chunk", batch=1, rows=256, capacity=4096, q_heads=32, kv_heads=8, head_dim=128, window=-1,
             dtype="bf16")
    return _case(c, name, kw)


def _self(name=None, **kw):
    c = dict(kind="self", train=False, batch=1, seq=512, q_heads=32, kv_heads=8, head_dim=128, mask="causal", window=-1,
             packed=False, bias=False, sink=False, dtype="bf16")
    return _case(c, name, kw)


def _case(c, name, kw):
    assert set(kw) <= set(c), set(kw) - set(c)
    c = dict(c, **kw)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # One conversation, a short context: the smallest call of the reference's decode benchmark.
        _decode("decode_one", batch=1, capacity=1024, shortest=1024, q_heads=8, kv_heads=8, dtype="f16"),
        # A small serving batch over a contiguous cache, grouped-query heads, every sequence at its own
        # length, a capacity that is no multiple of anything.
        _decode("decode_batch", batch=8, capacity=8190, shortest=2000, q_heads=32, kv_heads=8),
        # A loaded server: 64 sequences of 512 to 32768 tokens in a shared pool of 16-token pages.
        _decode("decode_paged", batch=64, capacity=32768, shortest=512, q_heads=32, kv_heads=8, page=16),
        # A sliding-window layer of such a server: long contexts in 64-token pages, of which a step sees
        # the last 4096 tokens.
        _decode("decode_window", batch=16, capacity=16384, shortest=1024, q_heads=64, kv_heads=8, page=64, window=4096),
        # Incremental prefill: the next 200 prompt tokens of two sequences, at two odd offsets into their caches.
        _chunk("chunk_prefill", batch=2, rows=200, capacity=8192),
        # The prefill of one short prompt.
        _self("prefill_short", batch=1, seq=512),
        # An ordinary prefill batch at head_dim 64 (a row of the reference's prefill benchmark).
        _self("prefill_d64", batch=2, seq=4096, q_heads=32, kv_heads=32, head_dim=64, dtype="f16"),
        # The training step of an 8B-parameter decoder layer's attention, sequence length 4096.
        _self("train_causal", train=True, batch=4, seq=4096),
        # Training on rows packed from several documents, under a sliding window.
        _self("train_packed", train=True, batch=8, seq=8192, q_heads=16, kv_heads=16, mask="window", window=4096, packed=True),
        # Training with a dense logit bias per head (relative positions) beside the causal mask.
        _self("train_bias", train=True, batch=2, seq=2048, q_heads=16, kv_heads=16, bias=True),
        # Training in float32 (a row of the reference's prefill benchmark).
        _self("train_f32", train=True, batch=2, seq=4096, q_heads=32, kv_heads=32, dtype="f32"),
        # Long-context training: one device's heads of a 32768-token sequence.
        _self("train_long", train=True, batch=1, seq=32768, q_heads=64, kv_heads=8),
    ]


HEADS = ((8, 8), (8, 1), (16, 16), (32, 32), (32, 8), (64, 8), (12, 4))


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng: random.Random):
    while True:
        c = _draw_one(rng)
        w = work(c)
        # no costlier than a listed case of the kind, and within what inputs of a few gigabytes hold
        most = {"decode": 9e9, "chunk": 9e9, "self": 9e9}[c["kind"]]
        if w["bytes"] <= most and w["flops"] <= (6e12 if c["dtype"] != "f32" else 2e12):
            return c


def _draw_one(rng):
    hq, hkv = rng.choice(HEADS)
    kind = rng.choice(("decode", "decode", "decode", "chunk", "self", "self", "train", "train", "train"))
    if kind == "decode":
        page = rng.choice((0, 0, 16, 32, 64, 128))
        capacity = _log_int(rng, 512, 131072 if page == 0 else 32768)
        if page:
            capacity = -(-capacity // page) * page
        batch = _log_int(rng, 1, 64)
        while batch > 1 and batch * capacity * hkv * 128 * 4 > 9e9:
            batch //= 2
        return _decode(batch=batch, capacity=capacity, shortest=max(1, int(capacity * rng.choice((0.02, 0.25, 0.5, 1.0)))),
                       q_heads=hq, kv_heads=hkv, head_dim=rng.choice((64, 80, 96, 128, 128, 128)), page=page,
                       window=rng.choice((-1, -1, -1, 1024, 4096)), dtype=rng.choice(("bf16", "bf16", "f16")))
    if kind == "chunk":
        capacity = 128 * _log_int(rng, 8, 256)
        return _chunk(batch=_log_int(rng, 1, 8), rows=_log_int(rng, 7, min(1024, capacity // 2)), capacity=capacity,
                      q_heads=hq, kv_heads=hkv, head_dim=rng.choice((64, 128, 128)),
                      window=rng.choice((-1, -1, -1, 1024)), dtype=rng.choice(("bf16", "bf16", "f16")))
    train = kind == "train"
    dtype = rng.choice(("bf16",) * 5 + ("f16",) * 2 + ("f32",))
    bias = dtype != "f32" and rng.random() < 0.2
    odd_dims = () if dtype == "f32" or bias else (80, 96)
    seq = 128 * _log_int(rng, 1, 16 if bias or dtype == "f32" else 128)
    mask = rng.choice(("causal",) * 4 + ("window", "none"))
    return _self(train=train, batch=_log_int(rng, 1, 8), seq=seq, q_heads=hq, kv_heads=hkv,
                 head_dim=rng.choice((64, 128, 128, 128) + odd_dims), mask=mask,
                 window=rng.choice((256, 1024, 4096)) if mask == "window" else -1,
                 packed=not bias and rng.random() < 0.3, bias=bias, sink=rng.random() < 0.15, dtype=dtype)


# ------------------------------------------------------------------------------------------- inputs


class State:
    """What a caller holds: the layer, the arguments of the call, and for training dO and the leaves."""

    def __init__(self, layer, args, insert=None, leaves=None, d_out=None):
        self.layer, self.args, self.insert, self.leaves, self.d_out = layer, args, insert, leaves, d_out


def _document_cuts(rng, seq):
    n = int(rng.integers(1, MAX_DOCS + 1))
    cuts = np.sort(rng.choice(np.arange(1, seq), size=min(n, seq - 1) - 1, replace=False)) if n > 1 else []
    return [0, *[int(x) for x in cuts], seq]


def _mask_bias(c, target, source):
    pos = dict(target_positions=target, source_positions=source)
    if c["window"] >= 0:
        return ab.SlidingWindowAttentionBias(ab.sliding_window_causal_mask(c["window"]), sliding_window_size=c["window"], **pos)
    return ab.CausalAttentionBias(**pos)


def prepare(c, seed):
    dev = torch.device("cuda:0")
    dtype = DTYPES[c["dtype"]]
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    rng = np.random.default_rng(int(seed))

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev, dtype=dtype)

    def positions(n):
        return torch.arange(n, device=dev, dtype=torch.int32)[None]

    b, hq, hkv, d = c["batch"], c["q_heads"], c["kv_heads"], c["head_dim"]
    layer = FlashAttention.default_config().set(softmax_scale=d ** -0.5).instantiate()
    if c["kind"] == "decode":
        lengths = rng.integers(c["shortest"], c["capacity"] + 1, size=b)
        last = torch.from_numpy(lengths.astype(np.int32) - 1).to(dev)[:, None]
        args = dict(q_proj=normal(b, 1, hq, d),
                    attention_logit_biases=ab.CompositeAttentionBias([_mask_bias(c, last, positions(c["capacity"]))]))
        if c["page"] == 0:
            return State(layer, dict(args, k_proj=normal(b, c["capacity"], hkv, d), v_proj=normal(b, c["capacity"], hkv, d),
                                     kv_cache_type=KVCache))
        pages = c["capacity"] // c["page"]
        pool = b * pages + 1    # page 0 is the padding page
        table = (torch.randperm(pool - 1, generator=gen, device=dev) + 1).to(torch.int32).reshape(b, pages)
        live = torch.from_numpy(-(-lengths // c["page"])).to(dev)
        table = torch.where(torch.arange(pages, device=dev)[None] < live[:, None], table, torch.zeros_like(table))
        k_pool, v_pool = normal(hkv, pool, c["page"], d), normal(hkv, pool, c["page"], d)
        insert = dict(k_proj=normal(b, 1, hkv, d), v_proj=normal(b, 1, hkv, d), key_positions=last)
        return State(layer, dict(args, k_proj=k_pool, v_proj=v_pool, page_indices=table, kv_cache_type=PagedKVCache), insert)
    if c["kind"] == "chunk":
        start = rng.integers(0, c["capacity"] - c["rows"] + 1, size=b).astype(np.int32)
        target = torch.from_numpy(start).to(dev)[:, None] + positions(c["rows"])
        bias = ab.CompositeAttentionBias([_mask_bias(c, target, positions(c["capacity"]))])
        return State(layer, dict(q_proj=normal(b, c["rows"], hq, d), k_proj=normal(b, c["capacity"], hkv, d),
                                 v_proj=normal(b, c["capacity"], hkv, d), attention_logit_biases=bias, kv_cache_type=KVCache))
    t = c["seq"]
    parts = []
    if c["mask"] != "none":
        parts.append(_mask_bias(c, positions(t), positions(t)))
    if c["packed"]:
        ids = np.ones((b, t), dtype=np.int32)
        for row in ids:
            for cut in _document_cuts(rng, t)[1:-1]:
                row[cut:] += 1
        parts.append(ab.SegmentIdAttentionBias(torch.from_numpy(ids).to(dev)))
    if c["bias"]:
        parts.append(ab.TensorAttentionBias.from_tensor(normal(1, hq, t, t)))
    args = dict(q_proj=normal(b, t, hq, d), k_proj=normal(b, t, hkv, d), v_proj=normal(b, t, hkv, d),
                attention_logit_biases=ab.CompositeAttentionBias(parts))
    if c["sink"]:
        args["logit_sink"] = torch.randn((hq,), generator=gen, device=dev, dtype=torch.float32)
    if not c["train"]:
        return State(layer, args)
    leaves = [args[name].requires_grad_(True) for name in ("q_proj", "k_proj", "v_proj", "logit_sink") if name in args]
    return State(layer, dict(args, is_training=True), leaves=leaves, d_out=normal(b, t, hq, d))


def run(s):
    if s.leaves is not None:
        out, _ = s.layer.compute_attention(**s.args)
        return [out, *torch.autograd.grad(out, s.leaves, s.d_out)]
    with torch.no_grad():
        if s.insert is None:
            return s.layer.compute_attention(**s.args)[0]
        k_pool, v_pool = paged_extend_step(s.args["k_proj"], s.args["v_proj"], s.args["page_indices"], **s.insert)
        return [s.layer.compute_attention(**s.args)[0], k_pool, v_pool]


# --------------------------------------------------------------------------------------------- work


def _pairs(lo, hi, window):
    """Visible (query, key) pairs of query positions lo .. hi-1 under a causal mask / sliding window."""
    q = np.arange(lo, hi, dtype=np.int64)
    return int((np.minimum(q, window) + 1 if window >= 0 else q + 1).sum())


def work(c):
    es = 4 if c["dtype"] == "f32" else 2
    b, hq, hkv, d = c["batch"], c["q_heads"], c["kv_heads"], c["head_dim"]
    if c["kind"] == "decode":
        mean = (c["shortest"] + c["capacity"]) / 2.0      # lengths are uniform in between
        if c["window"] >= 0:                              # of which a step sees the last window + 1
            n = np.arange(c["shortest"], c["capacity"] + 1)
            mean = float(np.minimum(n, c["window"] + 1).mean())
        new = 4 * b * hkv * d * es if c["page"] else 0    # the new token's rows, read and written
        return {"bytes": 2 * b * mean * hkv * d * es + 2 * b * hq * d * es + new, "flops": 4 * b * mean * hq * d}
    if c["kind"] == "chunk":
        # a chunk starts anywhere in the cache; on average in its middle
        start = (c["capacity"] - c["rows"]) // 2
        keys = start + c["rows"] if c["window"] < 0 else min(start + c["rows"], c["window"] + c["rows"])
        return {"bytes": 2 * b * keys * hkv * d * es + 2 * b * c["rows"] * hq * d * es,
                "flops": 4 * b * hq * d * _pairs(start, start + c["rows"], c["window"])}
    t = c["seq"]
    if c["packed"]:          # documents are drawn per row: the mean over many rows
        rng, rows, pairs = np.random.default_rng(0), 64, 0
        for _ in range(rows):
            cuts = _document_cuts(rng, t)
            for lo, hi in zip(cuts, cuts[1:]):
                pairs += (hi - lo) ** 2 if c["mask"] == "none" else _pairs(0, hi - lo, c["window"])
        pairs = b * pairs / rows
    else:
        pairs = b * (t * t if c["mask"] == "none" else _pairs(0, t, c["window"]))
    q_bytes, kv_bytes = b * t * hq * d * es, 2 * b * t * hkv * d * es
    bias = hq * (t * t if c["mask"] == "none" else _pairs(0, t, c["window"])) * es if c["bias"] else 0
    # the forward reads q, k, v and writes out; the backward reads those and dO and writes three gradients
    if not c["train"]:
        return {"bytes": 2 * q_bytes + kv_bytes + bias, "flops": 4 * hq * d * pairs}
    return {"bytes": 6 * q_bytes + 3 * kv_bytes + 2 * bias, "flops": 14 * hq * d * pairs}


def tolerance(c):
    # 16-bit: q, k, v are exact, P and dS are rounded to the element type ahead of their products and the
    # results at the end.  Against float64 arithmetic on the same inputs (256 to 2048 tokens; every mask,
    # packing, bias, sink; forward and gradients) the worst 2-norm error of an output is 0.0027 in bf16,
    # 0.00034 in f16 and 1.5e-6 in f32 (growing with the square root of the length), the worst single
    # element 0.095, 0.01 and 3.1e-5 of its size or the output's rms.  About four times that:
    return {
        "bf16": {"rel": 1.1e-2, "max": 0.35},
        "f16": {"rel": 1.4e-3, "max": 0.04},
        "f32": {"rel": 8e-6, "max": 2e-4},
    }[c["dtype"]]
