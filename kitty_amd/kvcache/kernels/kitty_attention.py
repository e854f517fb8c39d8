"""Decode attention over the packed cache with the reference's signature
(src/kitty/kvcache/kernels/kitty_attention.py:403-408): ``kitty_attention_forward(module, query,
kv_cache, scaling) -> (attn_output [B, 1, H_Q, D] fp16, None)``.

The reference runs a QK kernel, a torch softmax over a ``[B, H_Q, T]`` score tensor in HBM and an
SV kernel, each on a ``(B, H_KV)`` grid (:433-523).  Here one fused split-K kernel streams the
packed pages once (QK^T, online softmax and PV per split of the sequence) and a merge kernel
combines the splits; no score tensor exists.
"""
import functools
from typing import Optional

import torch
import torch.nn as nn

from ... import _lib
from ..utils_kv_per_layer import KVCache_Layer

MAX_KV_GROUP = 16   # kitty_attention.py:418


@functools.lru_cache(maxsize=4096)
def _split_plan(B: int, H_Q: int, H_KV: int, D: int, max_tiles: int, per_sequence: bool, num_splits: int):
    """(splits, workspace bytes) of a decode launch: a function of the sizes alone."""
    lib = _lib.lib()
    if num_splits <= 0:
        num_splits = lib.kitty_decode_attn_default_splits_d(B, H_KV, D, max_tiles, int(per_sequence))
    return num_splits, lib.kitty_decode_attn_workspace_bytes(B, H_Q, D, num_splits)


@functools.lru_cache(maxsize=4096)
def _chunk_split_plan(B: int, H_Q: int, H_KV: int, D: int, T_q: int, max_tiles: int):
    """(splits, workspace bytes) of a chunked-prefill launch: a function of the sizes alone."""
    lib = _lib.lib()
    num_splits = lib.kitty_prefill_attn_default_splits(B, H_Q, H_KV, D, T_q, max_tiles)
    return num_splits, lib.kitty_prefill_attn_workspace_bytes(B, H_Q, D, T_q, num_splits)


def kitty_attention_forward(
    module: nn.Module,
    query: torch.Tensor,
    kv_cache: KVCache_Layer,
    scaling: float,
    *,
    num_splits: Optional[int] = None,
    variant: int = 0,
):
    assert query.is_contiguous(), "Query tensor must be contiguous."
    B, H_Q, t_query, D = query.size()
    assert t_query == 1, "Only decoding step with t_query=1 is supported."
    assert H_Q == module.num_attention_heads, "H_Q must match num_attention_heads."
    H_KV = module.num_key_value_heads
    KV_GROUP = H_Q // H_KV
    assert KV_GROUP <= MAX_KV_GROUP, f"KV_GROUP ({KV_GROUP}) exceeds MAX_KV_GROUP ({MAX_KV_GROUP})."
    _lib.require_hip(query, "query")
    if query.dtype != torch.float16:
        raise ValueError(f"query must be float16, got {query.dtype}")
    if H_KV != kv_cache.H_KV or B > kv_cache.MAX_BS:
        raise ValueError("query does not match the cache (H_KV or batch size)")

    per_sequence = kv_cache.seq_counts is not None
    if per_sequence:
        max_tiles = 2 + kv_cache.MAX_PAGE
    else:
        max_tiles = 1 + (kv_cache.get_total_length() - kv_cache.Sink_Count + kv_cache.PAGE_SIZE - 1) // kv_cache.PAGE_SIZE
    num_splits, ws_bytes = _split_plan(B, H_Q, H_KV, D, max_tiles, per_sequence, num_splits or 0)
    ws = kv_cache.workspace(ws_bytes)
    # [B, T=1, H_Q, D], the layout HF attention modules expect (kitty_attention.py:475-481)
    attn_output = query.new_empty((B, t_query, H_Q, D))
    rc = _lib.lib().kitty_decode_attn(kv_cache.descriptor(), query.data_ptr(), B, H_Q, float(scaling),
                                      attn_output.data_ptr(), ws.data_ptr(), ws.numel(), num_splits, variant,
                                      _lib.current_stream_ptr(query.device))
    if rc:
        _lib.check(rc, "kitty_attention_forward")
    return attn_output, None


def kitty_prefill_attention(
    module: nn.Module,
    query: torch.Tensor,
    key_states: torch.Tensor,
    value_states: torch.Tensor,
    kv_cache: KVCache_Layer,
    scaling: float,
):
    """Chunked-prefill attention: ``query [B, H_Q, T_q, D]`` attends to everything ``kv_cache``
    holds and, causally, to the chunk's own ``key_states`` / ``value_states [B, H_KV, T_q, D]``
    (fp16, not yet appended).  Returns ``(attn_output [B, T_q, H_Q, D] fp16, None)``.

    An extension of the reference's interface, whose attention asserts ``t_query == 1``
    (kitty_attention.py:411) and whose prefill is dense attention on an empty cache
    (benchmark_kitty.py:302); cached tokens enter exactly as in decode.  Append the chunk afterwards
    with ``KittyCache.update`` (empty cache) or ``KittyCache.append``.
    """
    B, H_Q, T_q, D = query.size()
    assert H_Q == module.num_attention_heads, "H_Q must match num_attention_heads."
    H_KV = module.num_key_value_heads
    KV_GROUP = H_Q // H_KV
    assert KV_GROUP <= MAX_KV_GROUP, f"KV_GROUP ({KV_GROUP}) exceeds MAX_KV_GROUP ({MAX_KV_GROUP})."
    for name, t in (("query", query), ("key_states", key_states), ("value_states", value_states)):
        _lib.require_hip(t, name)
        if t.dtype != torch.float16:
            raise ValueError(f"{name} must be float16, got {t.dtype}")
    if key_states.shape != (B, H_KV, T_q, D) or value_states.shape != key_states.shape:
        raise ValueError(f"key_states / value_states must be [B, H_KV, T_q, D] = {(B, H_KV, T_q, D)}, got "
                         f"{tuple(key_states.shape)} / {tuple(value_states.shape)}")
    if H_KV != kv_cache.H_KV or B > kv_cache.MAX_BS:
        raise ValueError("query does not match the cache (H_KV or batch size)")
    if query.stride(-1) != 1:
        query = query.contiguous()
    if key_states.stride(-1) != 1:
        key_states = key_states.contiguous()
    if value_states.stride() != key_states.stride():
        value_states = value_states.contiguous()
        key_states = key_states.contiguous()

    attn_output = query.new_empty((B, T_q, H_Q, D))
    # tiles of the longest sequence (with counters on the device the host ints shadow it; any number of shares is right)
    max_tiles = 1 + kv_cache.PageCount_K + (kv_cache.Q_Buffer_Count_K > 0)
    num_splits, ws_bytes = _chunk_split_plan(B, H_Q, H_KV, D, T_q, max_tiles)
    # scratch of this call alone (128 MB at most, by the rule): torch's allocator hands the same block to the next layer
    ws = query.new_empty(ws_bytes, dtype=torch.uint8) if num_splits > 1 else None
    _launch_chunk(kv_cache.descriptor(), query, key_states, value_states, scaling, attn_output, ws, ws_bytes, num_splits,
                  "kitty_prefill_attention")
    return attn_output, None


def _launch_chunk(desc, query, key_states, value_states, scaling, out, ws, ws_bytes, num_splits, what: str) -> None:
    qs, ks = [x * 2 for x in query.stride()], [x * 2 for x in key_states.stride()]
    rc = _lib.lib().kitty_prefill_attn_split(desc, query.data_ptr(), qs[0], qs[1], qs[2], key_states.data_ptr(),
                                             value_states.data_ptr(), ks[0], ks[1], ks[2], query.shape[0], query.shape[1],
                                             query.shape[2], float(scaling), out.data_ptr(),
                                             None if ws is None else ws.data_ptr(), ws_bytes, num_splits,
                                             _lib.current_stream_ptr(query.device))
    if rc:
        _lib.check(rc, what)


def prompt_attention_ready(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, kv_cache: KVCache_Layer) -> bool:
    """The chunk kernel can run a prompt's dense causal attention on these tensors as they lie.  What stays with
    torch's attention: other types, devices and head dimensions (at 64 and 256 the kernel keeps fp32 probabilities
    and is slower than a dense kernel), rows off the 16-byte grid, autocast (which gives the result its type), and whatever
    is being differentiated or traced."""
    if not kv_cache.on_hip or kv_cache.D != 128 or kv_cache.MAX_PAGE < 1:
        return False
    B, H_Q, T, D = query.shape
    H = kv_cache.H_KV
    if key.shape != (B, H, T, 128) or value.shape != key.shape or D != 128 or H_Q % H or not 1 <= H_Q // H <= MAX_KV_GROUP \
            or not 1 <= T <= 1 << 24 or not 1 <= B <= 65535 or key.stride() != value.stride():
        return False
    if torch.compiler.is_compiling() or torch.is_autocast_enabled("cuda") or not _lib.launchable(kv_cache.KeyCache.device):
        return False
    grad = torch.is_grad_enabled()
    for x in (query, key, value):
        st = x.stride()
        if type(x) is not torch.Tensor or x.dtype != torch.float16 or x.device != kv_cache.KeyCache.device or (grad and x.requires_grad) \
                or st[3] != 1 or st[2] < 128 or st[0] % 8 or st[1] % 8 or st[2] % 8 or x.data_ptr() % 16:
            return False
    return True


def kitty_prompt_attention(query: torch.Tensor, key: torch.Tensor, value: torch.Tensor, kv_cache: KVCache_Layer,
                           scaling: float) -> torch.Tensor:
    """Dense causal attention of a prompt whose tensors pass ``prompt_attention_ready``: the chunk kernel over an empty
    cache.  It reads the kv heads in place (torch's dense attention takes them repeated per query head) and writes
    ``[B, T, H_Q, D]``, the layout the caller returns."""
    B, H_Q, T, D = query.shape
    out = query.new_empty((B, T, H_Q, D))
    num_splits, ws_bytes = _chunk_split_plan(B, H_Q, kv_cache.H_KV, D, T, 1)
    ws = query.new_empty(ws_bytes, dtype=torch.uint8) if num_splits > 1 else None
    _launch_chunk(kv_cache.empty_descriptor(), query, key, value, scaling, out, ws, ws_bytes, num_splits,
                  "kitty_prompt_attention")
    return out
