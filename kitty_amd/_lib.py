"""ctypes binding of libkitty_hip.so, the C-ABI library that holds every HIP kernel.

There is no fallback: if the library has not been built, or a tensor is not on a HIP device, the
callers raise.  Build it with ``python -m kitty_amd.build``.
"""
import ctypes
import os
from ctypes import POINTER, c_char_p, c_float, c_int, c_int32, c_int64, c_size_t, c_uint8, c_void_p

import torch
from torch.autograd import forward_ad

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(HERE, "libkitty_hip.so")
ABI_VERSION = 2
SEQ_COUNT_FIELDS = 8
STATUS_FIELDS = 4
# order of a status row (KITTY_STATUS_*, include/kitty_hip.h)
STATUS_NAMES = ("tokens_dropped", "flush_skipped", "bad_page_write", "bad_page_read")

# order of kitty_kv_layer.counts / seq_counts rows (include/kitty_hip.h)
CNT_SINK, CNT_PAGES_K, CNT_QBUF_K, CNT_PAGES_V, CNT_QBUF_V, CNT_LOCAL_V, CNT_LOCAL_OFF = range(7)


class KittyKVLayer(ctypes.Structure):
    """struct kitty_kv_layer (include/kitty_hip.h)."""
    _fields_ = [
        ("H_KV", c_int32), ("D", c_int32), ("D_BOOSTED", c_int32), ("PAGE_SIZE", c_int32),
        ("S", c_int32), ("MAX_PAGE", c_int32),
        ("counts", c_int32 * SEQ_COUNT_FIELDS),
        ("seq_counts", c_void_p),
        ("status", c_void_p),
        ("cache_pages_k", c_int64), ("cache_pages_v", c_int64),
        ("key_cache", c_void_p), ("key_cache_stride_page", c_int64),
        ("key_meta", c_void_p), ("key_meta_stride_page", c_int64),
        ("value_cache", c_void_p), ("value_cache_stride_page", c_int64),
        ("value_meta", c_void_p), ("value_meta_stride_page", c_int64),
        ("page_table_k", c_void_p), ("page_table_k_stride_b", c_int64),
        ("page_table_v", c_void_p), ("page_table_v_stride_b", c_int64),
        ("sink_k", c_void_p), ("sink_v", c_void_p),
        ("sink_stride_b", c_int64), ("sink_stride_h", c_int64),
        ("qbuf_k", c_void_p), ("qbuf_v", c_void_p), ("local_v", c_void_p),
        ("win_stride_b", c_int64), ("win_stride_h", c_int64),
    ]


_SIGNATURES = {
    "kitty_abi_version": (c_int, []),
    "kitty_last_error": (c_char_p, []),
    "kitty_select_boost_k": (c_int, [c_void_p, c_int64, c_int64, c_int64, c_int, c_int, c_int, c_int, c_int, c_int,
                                     c_int, c_int, c_void_p, c_void_p]),
    "kitty_quant_pack_k": (c_int, [c_void_p, c_int64, c_int64, c_int64, c_int, c_int, c_int, c_int, c_int, c_int,
                                   c_int, c_int, c_void_p, c_void_p, c_int64, c_int, c_void_p, c_int64, c_void_p,
                                   c_int64, c_int64, c_void_p, c_void_p]),
    "kitty_quant_pack_v": (c_int, [c_void_p, c_int64, c_int64, c_int64, c_int, c_int, c_int, c_int, c_int, c_int,
                                   c_int, c_void_p, c_int64, c_int, c_void_p, c_int64, c_void_p, c_int64, c_int64,
                                   c_void_p, c_void_p]),
    "kitty_decode_attn_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int]),
    "kitty_decode_attn_default_splits": (c_int, [c_int, c_int, c_int, c_int]),
    "kitty_decode_attn_default_splits_d": (c_int, [c_int, c_int, c_int, c_int, c_int]),
    "kitty_decode_attn_split": (c_int, [POINTER(KittyKVLayer), c_void_p, c_int, c_int, c_float, c_void_p, c_size_t,
                                        c_int, c_int, c_void_p]),
    "kitty_decode_attn_merge": (c_int, [c_void_p, c_size_t, c_int, c_int, c_int, c_int, c_void_p, c_void_p]),
    "kitty_profile_next_split": (c_int, [c_void_p, c_void_p]),
    "kitty_decode_attn": (c_int, [POINTER(KittyKVLayer), c_void_p, c_int, c_int, c_float, c_void_p, c_void_p,
                                  c_size_t, c_int, c_int, c_void_p]),
    "kitty_decode_attn_static": (c_int, [POINTER(KittyKVLayer), c_void_p, c_int, c_int, c_float, c_void_p, c_int, c_int,
                                         c_void_p]),
    "kitty_prefill_attn": (c_int, [POINTER(KittyKVLayer), c_void_p, c_int64, c_int64, c_int64, c_void_p, c_void_p,
                                   c_int64, c_int64, c_int64, c_int, c_int, c_int, c_float, c_void_p, c_void_p]),
    "kitty_prefill_attn_workspace_bytes": (c_size_t, [c_int, c_int, c_int, c_int, c_int]),
    "kitty_prefill_attn_default_splits": (c_int, [c_int, c_int, c_int, c_int, c_int, c_int]),
    "kitty_prefill_attn_split": (c_int, [POINTER(KittyKVLayer), c_void_p, c_int64, c_int64, c_int64, c_void_p, c_void_p,
                                         c_int64, c_int64, c_int64, c_int, c_int, c_int, c_float, c_void_p, c_void_p,
                                         c_size_t, c_int, c_void_p]),
    "kitty_append_token": (c_int, [POINTER(KittyKVLayer), c_void_p, c_void_p, c_int64, c_int64, c_void_p, c_void_p,
                                   c_int64, c_int, c_void_p]),
    "kitty_append_row": (c_int, [POINTER(KittyKVLayer), c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_int,
                                 c_void_p]),
    "kitty_flush_full": (c_int, [POINTER(KittyKVLayer), c_int, c_void_p]),
    "kitty_append_chunk": (c_int, [POINTER(KittyKVLayer), c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int, c_int,
                                   c_void_p]),
    "kitty_append_chunk_host": (c_int, [POINTER(KittyKVLayer), c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int,
                                        c_int, c_void_p]),
    "kitty_append_chunk_host_d": (c_int, [POINTER(KittyKVLayer), c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int,
                                          c_int, c_void_p]),
    "kitty_pack_prompt": (c_int, [POINTER(KittyKVLayer), c_int, c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int64,
                                  c_int64, c_int64, c_int, c_int, c_void_p]),
    "kitty_fake_quant_from": (c_int, [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int64, c_int64, c_int64, c_int, c_int,
                                      c_int, c_int, c_int, c_int, c_int, c_int, c_void_p]),
    "kitty_fake_quant_topk": (c_int, [c_void_p, c_int64, c_int64, c_int64, c_void_p, c_int64, c_int64, c_int64, c_int, c_int,
                                      c_int, c_int, c_int, c_int, c_int, c_int, c_void_p, c_int, c_int, c_void_p]),
    "kitty_sim_append": (c_int, [c_void_p, c_void_p, c_int64, c_int64, c_int64, c_int64, c_void_p, c_void_p, c_int64, c_int64,
                                 c_int64, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_int, c_void_p]),
    "kitty_fake_quant": (c_int, [c_void_p, c_int64, c_int64, c_int64, c_int, c_int, c_int, c_int, c_int, c_int,
                                 c_int, c_int, c_int, c_void_p, c_int64, c_int64, c_int64, c_int, c_void_p]),
}

EXPORTS = tuple(_SIGNATURES)
_lib = None


def lib() -> ctypes.CDLL:
    """The loaded library; raises if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise RuntimeError(
                f"{LIB_PATH} is missing: the HIP kernels are not built (run `python -m kitty_amd.build`). "
                "There is no CPU or PyTorch fallback for this path.")
        handle = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in _SIGNATURES.items():
            fn = getattr(handle, name)
            fn.restype, fn.argtypes = res, args
        if handle.kitty_abi_version() != ABI_VERSION:
            raise RuntimeError(f"libkitty_hip.so has ABI {handle.kitty_abi_version()}, expected {ABI_VERSION}")
        _lib = handle
    return _lib


def check(rc: int, what: str) -> None:
    """0 = ok; negative = argument rejected on the host (ValueError, as the reference's asserts and
    ValueErrors fire before launch); positive = hipError_t (RuntimeError)."""
    if rc == 0:
        return
    msg = lib().kitty_last_error().decode("utf-8", "replace")
    if rc < 0:
        raise ValueError(f"{what}: {msg} (code {rc})")
    raise RuntimeError(f"{what}: HIP error {rc}: {msg}")


def require_hip(t, name: str) -> None:
    if not t.is_cuda:
        raise RuntimeError(
            f"{name} lives on {t.device}; the Kitty kernels are HIP kernels for MI355X and there is no CPU path")


def launchable(device) -> bool:
    """A raw launch may stand in for tensor operations on ``device``: nothing records the operations (a jit trace,
    forward-mode AD; a kernel would be invisible to both) and raw launches go to that device, i.e. it is the current one.
    Callers look at gradients themselves."""
    # (no public question for "is a dual level active": without the name, tensor operations are always kept)
    return (getattr(forward_ad, "_current_level", 0) < 0 and not _is_tracing()
            and device.index in (None, _current_device()))


def current_stream_ptr(device) -> int:
    """Torch's current stream on ``device`` as a raw ``hipStream_t`` (the Stream object that
    ``torch.cuda.current_stream`` builds around it costs the host 1.5 us a call)."""
    if _raw_stream is None:
        return torch.cuda.current_stream(device).cuda_stream
    index = device.index
    return _raw_stream(_current_device() if index is None else index)


# the private names behind torch.cuda.current_stream, current_device and jit.is_tracing, where this build of torch has them
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)
_is_tracing = getattr(torch._C, "_is_tracing", torch.jit.is_tracing)
