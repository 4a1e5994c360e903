"""The host path in native code (csrc/host.cc): from a layer's tensors to the C ABI in one call.

Every function here answers None (`page_insert`: False) to a call that it does not take, and the caller goes on in Python:
what is refused, cast, copied or padded stays with the classes in `axlearn_amd.flash_attention` and with `axlearn_amd.ops`.
So does every call where the extension has not been built, or not for the torch that is there: Python does the same, slower."""

from __future__ import annotations

import importlib.util
import logging
import os

import torch  # the extension is linked against torch's libraries, which this loads

from axlearn_amd import _lib

PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_axl_host.so")

_module = None
_absent = False   # it did not load: said once, not tried again


def load():
    """The extension, with the classes it recognises; raises where it has not been built."""
    global _module
    if _module is None:
        from axlearn_amd import attention_bias as ab
        from axlearn_amd.kv_cache import KVCache, PagedKVCache

        if not os.path.exists(PATH):
            raise RuntimeError(f"{PATH} is missing. Build it with `make -C axlearn_amd/csrc`.")
        _lib.load()
        spec = importlib.util.spec_from_file_location("axlearn_amd._axl_host", PATH)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        if torch.__version__.split("+")[0] != module.torch_version:
            raise ImportError(f"{PATH} was built for torch {module.torch_version}, not for {torch.__version__}. "
                              "Build it again with `make -C axlearn_amd/csrc clean all`.")
        module.register_types(ab.CompositeAttentionBias, ab.CausalAttentionBias, ab.SlidingWindowAttentionBias,
                              ab.SegmentIdAttentionBias, ab.TensorAttentionBias, KVCache, PagedKVCache)
        _module = module
    return _module


def _loaded():
    """The extension, or None: then the calls take the way through Python, which needs the kernel library alone."""
    global _absent
    if _module is None and not _absent:
        try:
            load()
        except (RuntimeError, ImportError, OSError) as e:
            _absent = True
            logging.warning("Calls of the attention kernels go through Python, without the native host path: %s", e)
    return _module


def attend(q, k, v, bias, page_indices, kv_cache_type, logit_sink, softmax_scale, gpu_block_size):
    """(out, probs) of a call without anything to differentiate; (None, probs, mask_kind, window, segment_ids, dense bias)
    of one that needs an autograd node, its bias the caller's own tensor."""
    host = _module or _loaded()
    if host is None:
        return None
    return host.attend(q, k, v, bias, page_indices, kv_cache_type, logit_sink, softmax_scale, gpu_block_size, False)


def page_insert(k_pages, v_pages, k_proj, v_proj, page_indices, key_positions) -> bool:
    """Whether the new tokens [B,1,Hkv,D] were written into the pools."""
    host = _module or _loaded()
    return host is not None and host.page_insert(k_pages, v_pages, k_proj, v_proj, page_indices, key_positions, False) is True


def flash_fwd(q, k, v, segment_ids, logit_sink, softmax_scale, mask_kind, sliding_window, bias, bias_copy):
    """(out, lse)."""
    host = _module or _loaded()
    if host is None:
        return None
    return host.flash_fwd(q, k, v, segment_ids, logit_sink, softmax_scale, mask_kind, sliding_window, bias, bias_copy, False)


def flash_bwd(q, k, v, out, lse, d_out, segment_ids, logit_sink, softmax_scale, mask_kind, sliding_window, limit, bias):
    """(dq, dk, dv) or (dq, dk, dv, d_logit_sink), dS in the workspace where that applies and fits `limit` bytes."""
    host = _module or _loaded()
    if host is None:
        return None
    return host.flash_bwd(q, k, v, out, lse, d_out, segment_ids, logit_sink, softmax_scale, mask_kind, sliding_window, limit, bias,
                          False)
