"""Hugging Face attention-interface adapters.

Same entry points as the reference's ``cornstarch/kernel/interface.py``:
``create_bitfield_attention_mask`` (:13-30), ``cornstarch_attention_forward`` (:33-53, materialized
bool mask) and ``bitfield_attention_forward`` (:56-96).
"""

from __future__ import annotations

from typing import Optional

import torch
import torch.nn.functional as F
from torch import nn

import math

from . import _bam_hip
from ._bam_hip import host as _host
from .attention import flash_attn_func
from .bitfield_attention import _dtype_code, _kernel_ready, _padded_head_dim, _stream_ptr, bitfield_attn_func


def create_bitfield_attention_mask(input_ids: torch.Tensor, token_ids: dict[str, int] = {}) -> torch.Tensor:
    """int64 bitfields from token ids (format of the reference's interface.py:13-30): the n-th entry of
    ``token_ids`` (dict order) owns bit n + 1, carried by the tokens whose id equals its placeholder id;
    every other token is text: bit 62, bit 0 and the bits of all modalities, so that text attends,
    causally, to every modality."""
    bit_of = {name: 1 << (n + 1) for n, name in enumerate(token_ids)}
    text = (1 << 62) | 1 | sum(bit_of.values())
    bitfield = input_ids.new_full(input_ids.shape, text, dtype=torch.int64)
    for name, placeholder_id in token_ids.items():
        bitfield.masked_fill_(input_ids == placeholder_id, bit_of[name])
    return bitfield


def cornstarch_attention_forward(
    module: nn.Module,
    query: torch.Tensor,
    key: torch.Tensor,
    value: torch.Tensor,
    attention_mask: torch.Tensor,
    **kwargs,
) -> tuple[torch.Tensor, None]:
    """query (B, H, Sq, D), key/value (B, H, Sk, D), attention_mask bool (B, Sq, Sk)
    -> (attn_output (B, Sq, H, D), None); reference interface.py:33-53."""
    query = query.transpose(1, 2)
    key = key.transpose(1, 2)
    value = value.transpose(1, 2)
    attn_output = flash_attn_func(query, key, value, mask=attention_mask)
    return attn_output, None


def _decode_attention(query, key, value, scaling, dropout, sliding_window, softcap):
    """Single-token decode step of a model in eval mode: the new token attends to the cache, no bitfield is
    consulted.  The reference hands this case to the flash-attn CUDA package through transformers'
    ``flash_attention_forward`` with ``attention_mask=None``, forwarding ``scaling``, ``sliding_window`` and
    ``softcap`` (interface.py:71-83).  Here it is the decode kernel of the HIP library with the semantics that call
    has for one query at the last position: ``scaling`` (default 1/sqrt(D)) multiplies q.k, ``softcap`` turns a
    score s into softcap * tanh(s / softcap), ``sliding_window`` (when the cache is longer than it) keeps the last
    ``sliding_window`` keys.  Dropout is inactive in eval mode either way.

    query (B, Hq, 1, D), key / value (B, Hkv, Sk, D) -> (B, 1, Hq, D) in the dtype of query."""
    if not dropout and (sliding_window is None or sliding_window > 0) and (softcap is None or softcap >= 0):
        out = _host.decode(query, key, value, scaling, sliding_window or 0, softcap or 0.0)
        if out is not None:
            return out, None
    # the general path: other layouts and head dims, and what is refused
    batch, nheads, q_len, d = query.shape
    _, nheads_k, seqlen_k, _ = key.shape
    assert q_len == 1
    assert query.is_cuda and key.is_cuda and value.is_cuda, "bitfield attention runs on the GPU only"
    assert query.dtype == key.dtype == value.dtype and query.dtype in (torch.float16, torch.bfloat16)
    assert key.shape == value.shape and key.shape[0] == batch and key.shape[3] == d and nheads % nheads_k == 0
    assert d <= 128, "FlashAttention only support head dimensions up to 128"
    if dropout:
        raise NotImplementedError("bitfield attention decode step: dropout is not supported (eval mode passes 0.0)")
    if sliding_window is not None and sliding_window <= 0:
        raise ValueError(f"sliding_window must be positive, got {sliding_window}")
    if softcap is not None and softcap < 0:
        raise ValueError(f"softcap must not be negative, got {softcap}")
    scale = float(scaling) if scaling is not None else 1.0 / math.sqrt(d)

    q, k, v = query.transpose(1, 2), key.transpose(1, 2), value.transpose(1, 2)  # (B, S, H, D) views
    dp = _padded_head_dim(d)
    if dp != d:  # zero columns change neither q.k nor the first d columns of p.v
        q, k, v = (F.pad(x, (0, dp - d)) for x in (q, k, v))
    q = q if q.stride(-1) == 1 else q.contiguous()
    k, v = _kernel_ready(k, 8), _kernel_ready(v, 8)
    out = torch.empty((batch, 1, nheads, dp), dtype=query.dtype, device=query.device)
    window = int(sliding_window or 0)
    with torch.cuda.device(query.device):
        # the keys are split over many workgroups; their partial results meet in a small workspace
        ws_bytes = _bam_hip.load().bam_decode_workspace_bytes(batch, seqlen_k, nheads, nheads_k, dp, window)
        ws = torch.empty((ws_bytes,), dtype=torch.uint8, device=query.device) if ws_bytes > 0 else None
        _bam_hip.call(
            "bam_decode", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(),
            q.stride(0), q.stride(2), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2),
            out.stride(0), out.stride(2), batch, seqlen_k, nheads, nheads_k, dp, scale, _dtype_code(query.dtype),
            window, float(softcap or 0.0), ws.data_ptr() if ws is not None else None, ws_bytes,
            _stream_ptr(query.device),
        )
    if dp != d:
        out = out[..., :d].contiguous()
    return out, None


def bitfield_attention_forward(
    module: nn.Module,
    query: torch.Tensor,
    key: torch.Tensor,
    value: torch.Tensor,
    attention_mask: torch.Tensor,
    dropout: float = 0.0,
    scaling: Optional[float] = None,
    sliding_window: Optional[int] = None,
    softcap: Optional[float] = None,
    **kwargs,
) -> tuple[torch.Tensor, None]:
    """query (B, Hq, S, D), key/value (B, Hkv, S, D), attention_mask int64 (B, S)
    -> (attn_output (B, S, Hq, D), None).

    As in the reference, ``scaling``, ``dropout``, ``sliding_window`` and ``softcap`` are
    not forwarded to the bitfield kernel, which always uses 1/sqrt(D) (interface.py:94); the
    single-token decode step of a model in eval mode does honour them (interface.py:71-83)."""
    if not module.training and query.shape[2] == 1:
        return _decode_attention(query, key, value, scaling, dropout, sliding_window, softcap)

    assert (
        attention_mask is not None and attention_mask.dtype == torch.int64
    ), "Bitfield attention requires an attention mask of type torch.int64."

    query = query.transpose(1, 2)
    key = key.transpose(1, 2)
    value = value.transpose(1, 2)

    attn_output = bitfield_attn_func(query, key, value, bitfield_mask=attention_mask)
    return attn_output, None


def register_bitfield_attention(name: str = "bitfield_attention") -> None:
    """Register the adapter in transformers' attention registry, as the reference does at
    import time (cornstarch/models/multimodal_language_model/modeling_multimodal_language_model.py:42)."""
    from transformers.modeling_utils import ALL_ATTENTION_FUNCTIONS

    ALL_ATTENTION_FUNCTIONS.update({name: bitfield_attention_forward})
