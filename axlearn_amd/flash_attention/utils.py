"""Kernel dispatch: first supported candidate wins.

Mirrors axlearn/common/flash_attention/utils.py:31-163.  Only the "gpu" backend has candidates
here: this package is the MI355X kernel path and carries no CPU / XLA / TPU implementation, so every
other backend name yields None, which the calling layer treats as "use standard attention"
(axlearn/common/flash_attention/layer.py:278-285).
"""

from __future__ import annotations

import logging
from typing import Any, Optional

from axlearn_amd.attention_bias import BaseAttentionBias
from axlearn_amd.flash_attention.attention_types import FlashAttentionWithShardMapSpecs
from axlearn_amd.flash_attention.common import Tensor
from axlearn_amd.flash_attention.hip_attention import HipFlashAttention
from axlearn_amd.flash_attention.hip_decoding import HipDecoding, HipPagedAttention
from axlearn_amd.kv_cache import BaseKVCache, PagedKVCache

BACKENDS = dict(
    # Inference kernels are tried first, then the training / prefill kernel.
    gpu=[HipDecoding, HipFlashAttention],
)
PAGED_ATTN_BACKENDS = dict(
    gpu=[HipPagedAttention],
)


def flash_attention_implementation(
    backend: str,
    *,
    query: Tensor,
    key: Tensor,
    value: Tensor,
    bias: BaseAttentionBias,
    logit_sink: Optional[Tensor] = None,
    softmax_scale: float = 1.0,
    kv_cache_type: Optional[type[BaseKVCache]] = None,
    tpu_block_size: int = 512,
    gpu_block_size: int = 128,
    dropout_rate: Optional[float] = 0.0,
    page_tables: Optional[Tensor] = None,
    backend_overrides: Optional[dict[str, Any]] = None,
) -> Optional[FlashAttentionWithShardMapSpecs]:
    """Returns the first kernel of `backend` that supports the request, or None.

    query [B,T,Hq,D]; key/value [B,S,Hkv,D], or page pools [Hkv,pages,page_size,D] together with
    page_tables [B,pages_per_sequence] when kv_cache_type is PagedKVCache.
    """
    if dropout_rate is None:
        dropout_rate = 0.0
    candidates = BACKENDS.get(backend, [])
    if kv_cache_type == PagedKVCache:
        candidates = PAGED_ATTN_BACKENDS.get(backend, [])
    common_cfg = dict(
        dropout_rate=dropout_rate,
        interpret=_interpret(backend),
        softmax_scale=softmax_scale,
        tpu_block_size=tpu_block_size,
        gpu_block_size=gpu_block_size,
        backend_overrides=backend_overrides,
    )
    input_batch = dict(
        query=query, key=key, value=value, page_tables=page_tables, bias=bias, logit_sink=logit_sink
    )
    for klass in candidates:
        if not klass.serves(query, kv_cache_type):
            continue
        attn_fn = klass.default_config().set(**common_cfg).instantiate()
        if attn_fn.is_supported(input_batch=input_batch, kv_cache_type=kv_cache_type):
            logging.info("Using %s for flash attention.", attn_fn.name())
            return attn_fn.build(input_batch=input_batch)
    logging.warning("Using standard attention as flash attention fallback.")
    return None


def _interpret(backend: str) -> bool:
    return backend == "cpu"
