"""The native host path (csrc/host.cc) against the way through Python: the same parameter blocks, and no call taken that the
Python classes refuse, copy, cast or pad for."""

import ctypes
import logging
import random

import pytest
import torch
from torch.autograd import forward_ad

from axlearn_amd import _host, _lib, ops
from axlearn_amd import attention_bias as ab
from axlearn_amd.flash_attention.layer import FlashAttention
from axlearn_amd.kv_cache import KVCache, PagedKVCache, paged_extend_step

OUTPUTS = ("out", "lse", "dq", "dk", "dv", "d_logit_sink", "workspace", "workspace_bytes")
BLOCKS = dict(axl_decode=_lib.AxlDecodeParams, axl_paged_decode=_lib.AxlPagedDecodeParams, axl_flash_chunk=_lib.AxlFlashChunkParams,
              axl_flash_fwd=_lib.AxlFlashFwdParams, axl_flash_bwd_phases=_lib.AxlFlashBwdParams,
              axl_paged_kv_insert=_lib.AxlPageInsertParams)


def _fields(block):
    """A parameter block as nested plain values, but for what the call allocates."""
    def plain(x):
        return {n: plain(getattr(x, n)) for n, _ in x._fields_} if isinstance(x, ctypes.Structure) else x

    return {n: v for n, v in plain(block).items() if n not in OUTPUTS}


@pytest.fixture
def recorded(monkeypatch):
    """CPU tensors pass for the GPU's; the list of blocks that reach the C ABI."""
    real, seen = _lib.load(), []

    class Recorder:
        def __getattr__(self, name):
            if name not in BLOCKS:
                return getattr(real, name)
            return lambda p, *rest: seen.append(_fields(p._obj)) or 0

    monkeypatch.setattr(_lib, "load", lambda: Recorder())
    monkeypatch.setattr(_lib, "current_stream_ptr", lambda: 0)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(ops, "_device_properties", lambda device: (288 << 30, 256))
    return seen


def _without_native_calls(monkeypatch):
    for name in ("attend", "flash_fwd", "flash_bwd"):
        monkeypatch.setattr(_host, name, lambda *a: None)
    monkeypatch.setattr(_host, "page_insert", lambda *a: False)


@pytest.fixture
def through_python(monkeypatch, recorded):
    """Calls go through Python on CPU tensors that pass for the GPU's; the list of blocks that reach the C ABI."""
    _without_native_calls(monkeypatch)
    logging.disable(logging.WARNING)
    yield recorded
    logging.disable(logging.NOTSET)


def _native(cls, name, *args):
    """What the native path would hand to the C ABI, as `_fields`, or None."""
    block = getattr(_host.load(), name)(*args, True)
    assert block is None or len(block) == ctypes.sizeof(cls)
    return None if block is None else _fields(cls.from_buffer_copy(block))


def _same(seen, got, bias=None):
    assert len(seen) == 1
    for x in (seen[0], got):
        if bias is not None and bias.dtype == torch.float16:
            x["aux"] = dict(x["aux"], bias=None)    # an fp32 copy of each way's own
    assert seen[0] == got


def _view(rng, shape, dtype):
    """A tensor of `shape`: dense, heads ahead of rows, a part of a larger one, at an odd offset, or not dense in its rows."""
    b, t, h, d = shape
    kind = rng.choice(("dense",) * 30 + ("heads", "slice", "offset", "columns"))
    if kind == "heads":
        return torch.zeros(b, h, t, d, dtype=dtype).transpose(1, 2)
    if kind == "slice":
        return torch.zeros(b, t + 3, h + 1, d + 8, dtype=dtype)[:, 1:t + 1, :h, :d]
    if kind == "offset":
        return torch.zeros(b * t * h * d + 1, dtype=dtype)[1:].view(shape)
    if kind == "columns":
        return torch.zeros(b, t, h, 2 * d, dtype=dtype)[..., ::2]
    return torch.zeros(shape, dtype=dtype)


def _positions(rng, b, t):
    dtype = rng.choice((torch.int32,) * 5 + (torch.int64,) * 5 + (torch.int16,))
    x = torch.arange(t + 2, dtype=dtype)[None, 1:t + 1]
    if rng.random() < 0.6 and b > 1:
        x = x.repeat(b, 1) if rng.random() < 0.7 else torch.zeros(t, b, dtype=dtype).t()
    return x


def _bias(rng, b, t, s, hq, segments):
    pos = dict(target_positions=_positions(rng, b, t), source_positions=torch.arange(s)[None])
    causal = ab.CausalAttentionBias(**pos)
    window = rng.choice((0, 5, 4096))
    sliding = ab.SlidingWindowAttentionBias(ab.sliding_window_causal_mask(window), sliding_window_size=window, **pos)
    ids = torch.zeros(b if rng.random() < 0.9 else b + 1, t, dtype=rng.choice((torch.int32,) * 4 + (torch.int64,)))
    dense = torch.zeros(rng.choice((1, 1, b, b + 1)), rng.choice((1, hq, hq)), t, s, dtype=rng.choice((torch.float32, torch.bfloat16, torch.float16)))
    dense = rng.choice([dense] * 6 + [dense.new_zeros(*dense.shape[:2], s, t).transpose(2, 3), dense.expand(b, -1, -1, -1) if len(dense) == 1 else dense])
    other = rng.choice([None] * 24 + [ab.TensorAttentionBias(dense)] * 6 + [ab.ZeroAttentionBias(),
                                      ab.TensorAttentionBias(torch.zeros(1, hq, t, s), dtype=torch.bfloat16),
                                      ab.MaskFnAttentionBias(ab.causal_mask, **pos), causal, "none"])
    members = rng.choice(([causal], [sliding], [causal], [sliding], [causal], [sliding], [], [causal, sliding]))
    members = members + ([ab.SegmentIdAttentionBias(ids)] if segments and rng.random() < 0.5 else [])
    members = members + ([None] if other == "none" else [other] if other is not None else [])
    rng.shuffle(members)
    if len(members) == 1 and members[0] is not None and rng.random() < 0.3:
        return members[0]
    return ab.CompositeAttentionBias(tuple(members) if rng.random() < 0.2 else members)


def _layer_call(rng):
    kind = rng.choice(("decode", "paged", "chunk", "self", "self"))
    b, hkv = rng.choice((1, 2, 3)), rng.choice((1, 2))
    hq, d = hkv * rng.choice((1, 4)), rng.choice((64, 128, 64, 128, 64, 128, 80, 72, 96, 24, 36, 136))
    dtype = rng.choice((torch.bfloat16, torch.float16, torch.float32))
    t = 1 if kind in ("decode", "paged") else rng.choice((7, 128)) if kind == "chunk" else rng.choice((128, 256, 256, 256, 200))
    s = t if kind == "self" and rng.random() < 0.8 else rng.choice((256, 384, 512, 200))
    kv_dtype = dtype if rng.random() < 0.95 else torch.bfloat16
    args = dict(q_proj=_view(rng, (b, t, hq, d), dtype))
    if kind == "paged":
        page = rng.choice((16, 32, 64, 128, 16, 32, 8, 24))
        args.update({n: _view(rng, (hkv, 5, page, d), kv_dtype) for n in ("k_proj", "v_proj")})
        args["page_indices"] = torch.zeros(b, 3, dtype=rng.choice((torch.int32,) * 5 + (torch.int64,)))
        s = 3 * page
    else:
        args.update({n: _view(rng, (b, s, hkv, d), kv_dtype) for n in ("k_proj", "v_proj")})
        if rng.random() < 0.05:
            args["v_proj"] = args["v_proj"][:, :-1]
    args["kv_cache_type"] = dict(decode=KVCache, paged=PagedKVCache, chunk=KVCache).get(kind)
    args["attention_logit_biases"] = _bias(rng, b, t, s, hq, kind == "self")
    if rng.random() < 0.15:
        args["logit_sink"] = torch.zeros(hq, dtype=rng.choice((torch.float32, torch.bfloat16)))
    return rng.choice((0.125, 1.0) * 8 + (-1.0,)), args


@pytest.mark.parametrize("seed", range(6))
def test_layer_calls_reach_the_kernels_with_the_same_blocks(through_python, seed):
    rng, taken, refused = random.Random(seed), 0, 0
    for _ in range(250):
        scale, args = _layer_call(rng)
        layer = FlashAttention.default_config().set(softmax_scale=scale).instantiate()
        through_python.clear()
        try:
            with torch.no_grad():
                out, probs = layer.compute_attention(**args)
        except Exception:  # pylint: disable=broad-except
            through_python.clear()
            refused += 1
        cls = {KVCache: _lib.AxlDecodeParams if args["q_proj"].shape[1] == 1 else _lib.AxlFlashChunkParams,
               PagedKVCache: _lib.AxlPagedDecodeParams}.get(args["kv_cache_type"], _lib.AxlFlashFwdParams)
        got = _native(cls, "attend", args["q_proj"], args["k_proj"], args["v_proj"], args["attention_logit_biases"],
                      args.get("page_indices"), args["kv_cache_type"], args.get("logit_sink"), scale, 128)
        if got is not None:
            taken += 1
            members = getattr(args["attention_logit_biases"], "biases", ())
            dense = [m._internal_value for m in members if type(m) is ab.TensorAttentionBias]
            _same(through_python, got, *dense)
            assert probs.shape == (args["q_proj"].shape[0], args["q_proj"].shape[2], args["q_proj"].shape[1], probs.shape[3])
    assert taken > 20 and refused > 20, (taken, refused)


@pytest.mark.parametrize("seed", range(4))
def test_forward_and_backward_reach_the_kernels_with_the_same_blocks(through_python, seed):
    rng, taken = random.Random(seed), 0
    for _ in range(150):
        b, hkv, d, t = rng.choice((1, 2)), rng.choice((1, 8)), rng.choice((64, 128, 96, 80)), rng.choice((128, 256, 1024))
        hq, s = hkv * rng.choice((1, 4)), t if rng.random() < 0.9 else t + 128
        dtype = rng.choice((torch.bfloat16, torch.float16, torch.float32))
        q, do, out = (_view(rng, (b, t, hq, d), dtype) for _ in range(3))
        k, v = (_view(rng, (b, s, hkv, d), dtype) for _ in range(2))
        seg = torch.zeros(b, t, dtype=rng.choice((torch.int32, torch.int64))) if rng.random() < 0.4 else None
        sink = torch.zeros(hq, dtype=rng.choice((torch.float32, torch.bfloat16))) if rng.random() < 0.2 else None
        kind, window, limit = rng.choice((0, 1, 2)), rng.choice((0, 300)), rng.choice((0, 1 << 20, 1 << 34))
        lse = torch.zeros(b, hq, t)
        bias = None
        if rng.random() < 0.4 and t <= 256:
            bias = torch.zeros(rng.choice((1, b)), rng.choice((1, hq)), t, s, dtype=rng.choice((torch.float32, torch.bfloat16, torch.float16)))
            bias = rng.choice((bias, bias, bias, bias.new_zeros(*bias.shape[:3], s + 8)[..., :s], bias.new_zeros(*bias.shape[:2], s, t).transpose(2, 3)))
        copy = torch.empty(bias.shape, dtype=bias.dtype) if bias is not None and rng.random() < 0.4 else None
        kw = dict(softmax_scale=0.5, mask_kind=kind, sliding_window=window, segment_ids=seg, logit_sink=sink, bias=bias)
        for name, cls, call, args in (
                ("flash_fwd", _lib.AxlFlashFwdParams, lambda: ops.flash_fwd(q, k, v, bias_copy=copy, **kw),
                 (q, k, v, seg, sink, 0.5, kind, window, bias, copy)),
                ("flash_bwd", _lib.AxlFlashBwdParams,
                 lambda: ops.flash_bwd(q, k, v, out, lse, do, ds_workspace=None, ds_workspace_limit=limit, **kw),
                 (q, k, v, out, lse, do, seg, sink, 0.5, kind, window, limit, bias))):
            through_python.clear()
            try:
                call()
            except Exception:  # pylint: disable=broad-except
                through_python.clear()
            got = _native(cls, name, *args)
            if got is not None:
                taken += 1
                _same(through_python, got, bias)
    assert taken > 60


def test_page_inserts_reach_the_kernel_with_the_same_block(through_python):
    rng, taken = random.Random(0), 0
    for _ in range(200):
        b, hkv, d, page = rng.choice((1, 3)), rng.choice((1, 2)), rng.choice((64, 128)), rng.choice((16, 64))
        dtype = rng.choice((torch.bfloat16, torch.float16, torch.float32))
        k_pool, v_pool = (_view(rng, (hkv, 4, page, d), dtype) for _ in range(2))
        k, v = (_view(rng, (b, 1, hkv, d), dtype if rng.random() < 0.9 else torch.float32) for _ in range(2))
        table = torch.zeros(b, 2, dtype=rng.choice((torch.int32,) * 4 + (torch.int64,)))
        pos = torch.zeros(rng.choice((1, b)), 1, dtype=rng.choice((torch.int32,) * 4 + (torch.int64,)))
        through_python.clear()
        try:
            paged_extend_step(k_pool, v_pool, table, k_proj=k, v_proj=v, key_positions=pos)
        except Exception:  # pylint: disable=broad-except
            through_python.clear()
        got = _native(_lib.AxlPageInsertParams, "page_insert", k_pool, v_pool, k, v, table, pos)
        if got is not None:
            taken += 1
            assert through_python == [got]
    assert taken > 40


def test_calls_that_something_looks_at_by_its_operations_go_through_python():
    x = torch.zeros(1, 128, 1, 64)
    bias = ab.CompositeAttentionBias([])

    def taken(q=x):
        return _host.load().attend(q, x, x, bias, None, None, None, 0.125, 128, True) is not None

    class Subclass(torch.Tensor):
        pass

    assert taken() and taken(torch.nn.Parameter(x))
    assert not taken(x.as_subclass(Subclass))
    assert not taken(x.to_sparse())
    seen = []
    torch.func.vmap(lambda q: seen.append(taken(q)) or q)(x[None])
    torch.func.grad(lambda q: seen.append(taken(q)) or q.sum())(x)
    torch.jit.trace(lambda q: seen.append(taken(q)) or q + 1, x, check_trace=False)
    with forward_ad.dual_level():
        seen.append(taken())
    with torch.device("cpu"):        # a mode of torch functions
        seen.append(taken())
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode():
        seen.append(taken())
    assert seen and not any(seen)
    assert taken()
    assert _host.load().attend(x, x, x, bias, None, None, None, 0.125, 128, False) is None   # not on the GPU


def _no_extension(monkeypatch, tmp_path, how):
    monkeypatch.setattr(_host, "_module", None)
    monkeypatch.setattr(_host, "_absent", False)
    if how == "missing":
        monkeypatch.setattr(_host, "PATH", str(tmp_path / "_axl_host.so"))
    elif how == "not a library":
        (tmp_path / "_axl_host.so").write_bytes(b"\x7fELF")
        monkeypatch.setattr(_host, "PATH", str(tmp_path / "_axl_host.so"))
    elif how == "another torch":
        monkeypatch.setattr(torch, "__version__", "1.13.0+rocm5.2")
    else:
        def load():
            raise RuntimeError("libaxl_attn_hip.so is missing.")
        monkeypatch.setattr(_lib, "load", load)


@pytest.mark.parametrize("how", ["missing", "not a library", "another torch"])
def test_without_the_extension_calls_reach_the_kernels_through_python(monkeypatch, tmp_path, caplog, recorded, how):
    """The extension is not there, or does not load here: every call takes the way through Python, which says so once."""
    _no_extension(monkeypatch, tmp_path, how)
    with pytest.raises((RuntimeError, ImportError)):
        _host.load()
    x, pool = torch.zeros(1, 128, 2, 64, dtype=torch.bfloat16), torch.zeros(2, 4, 16, 64, dtype=torch.bfloat16)
    layer = FlashAttention.default_config().set(softmax_scale=0.125).instantiate()
    q = x.clone().requires_grad_(True)
    with caplog.at_level(logging.WARNING):
        out, _ = layer.compute_attention(q_proj=q, k_proj=x, v_proj=x, attention_logit_biases=ab.CompositeAttentionBias([]))
        out.backward(x)
        paged_extend_step(pool, pool.clone(), torch.zeros(1, 2, dtype=torch.int32), k_proj=x[:, :1], v_proj=x[:, :1],
                          key_positions=torch.zeros(1, 1, dtype=torch.int32))
    assert len(recorded) == 3 and q.grad.shape == q.shape   # forward, backward, insert
    assert len([r for r in caplog.records if "host path" in r.getMessage()]) == 1


@pytest.mark.parametrize("how", ["missing", "another torch", "no kernel library"])
def test_without_libraries_what_needs_none_is_answered(monkeypatch, tmp_path, how):
    """A request that no kernel supports goes to the fallback, and sizes that do not fit together are refused in Python."""
    _no_extension(monkeypatch, tmp_path, how)
    layer = FlashAttention.default_config().set(softmax_scale=0.125).instantiate()
    x = torch.zeros(1, 100, 2, 64)
    call = lambda k, **kw: layer.compute_attention(q_proj=x, k_proj=k, v_proj=k, attention_logit_biases=ab.CompositeAttentionBias([]), **kw)
    answer = (torch.ones(1), None)
    assert call(x, fallback=lambda **kw: answer) is answer
    with pytest.raises(ValueError):
        call(torch.zeros(2, 100, 2, 64))
    with pytest.raises(ValueError):
        paged_extend_step(x, x, torch.zeros(1, 2, dtype=torch.int32), k_proj=x, v_proj=x[:, :1], key_positions=torch.zeros(1, 1))


def test_backward_by_the_size_rule_refuses_cpu_tensors_as_the_other_calls_do():
    x, lse = torch.zeros(1, 128, 2, 64, dtype=torch.bfloat16), torch.zeros(1, 2, 128)
    with pytest.raises(_lib.AxlError, match="must live on the GPU"):
        ops.flash_bwd(x, x, x, x, lse, x, ds_workspace=None)
    with pytest.raises(_lib.AxlError, match="does not match"):   # sizes first, whatever the device
        ops.flash_bwd(x, x[..., :32], x, x, lse, x, mask_kind=ops.MASK_CAUSAL, ds_workspace=None)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["decode", "paged", "chunk", "self", "train", "train_bias", "train_bias_f16"])
def test_native_calls_give_the_bits_of_those_through_python(kind, monkeypatch):
    """On a stream of their own, each behind work that its inputs wait for; every step of them native, and none of those through
    Python."""
    gen = torch.Generator("cuda").manual_seed(0)
    b, hq, hkv, d, s = 2, 8, 2, 128, 512
    t = dict(decode=1, paged=1, chunk=40).get(kind, s)
    r = lambda *shape: torch.randn(shape, generator=gen, device="cuda").bfloat16()
    target = (torch.arange(t, device="cuda")[None] + torch.tensor([[s - t], [100 if t < s else 0]], device="cuda")).int()
    bias = ab.CompositeAttentionBias([ab.CausalAttentionBias(target_positions=target, source_positions=torch.arange(s, device="cuda")[None])])
    if kind.startswith("train_bias"):
        bias.biases.append(ab.TensorAttentionBias.from_tensor(r(1, hq, t, s).to(torch.float16 if kind.endswith("f16") else torch.bfloat16)))
    args = dict(q_proj=r(b, t, hq, d), attention_logit_biases=bias)
    pools = [r(hkv, 40, 16, d) for _ in range(2)]
    new = dict(k_proj=r(b, 1, hkv, d), v_proj=r(b, 1, hkv, d), key_positions=target[:, -1:].contiguous())
    if kind == "paged":
        args["page_indices"] = (torch.randperm(39, generator=gen, device="cuda")[None].repeat(b, 1)[:, :32] + 1).int().contiguous()
        args["kv_cache_type"] = PagedKVCache
    else:
        args.update(k_proj=r(b, s, hkv, d), v_proj=r(b, s, hkv, d))
        args["kv_cache_type"] = KVCache if kind in ("decode", "chunk") else None
    d_out, sink = r(b, t, hq, d), torch.randn(hq, generator=gen, device="cuda")
    layer = FlashAttention.default_config().set(softmax_scale=d ** -0.5).instantiate()

    def call():
        x = {n: v.clone() if isinstance(v, torch.Tensor) else v for n, v in args.items()}
        if kind == "paged":
            k, v = (p.clone() for p in pools)
            k, v = paged_extend_step(k, v, x["page_indices"], **new)
            with torch.no_grad():
                return [layer.compute_attention(**x, k_proj=k, v_proj=v)[0], k, v]
        if not kind.startswith("train"):
            return [layer.compute_attention(**x)[0]]
        leaves = [x[n].requires_grad_(True) for n in ("q_proj", "k_proj", "v_proj")] + [sink.clone().requires_grad_(True)]
        out, _ = layer.compute_attention(**x, logit_sink=leaves[3], is_training=True)
        return [out, *torch.autograd.grad(out, leaves, d_out)]

    torch.cuda.synchronize()
    side, taken = torch.cuda.Stream(), []

    def noted(name, native):
        def f(*a):
            result = native(*a)
            if result is not None and result is not False:
                taken.append(name)
            return result
        return f

    with monkeypatch.context() as m:
        for name in ("attend", "flash_fwd", "flash_bwd", "page_insert"):
            m.setattr(_host, name, noted(name, getattr(_host, name)))
        with torch.cuda.stream(side):
            got = [call() for _ in range(3)]
        side.synchronize()
    steps = dict(paged=["page_insert", "attend"]).get(kind, ["attend", "flash_fwd", "flash_bwd"] if kind.startswith("train") else ["attend"])
    assert taken == 3 * steps
    with monkeypatch.context() as m:
        _without_native_calls(m)
        want = call()
    torch.cuda.synchronize()
    for outs in got:
        assert all(torch.equal(x, y) for x, y in zip(outs, want))
