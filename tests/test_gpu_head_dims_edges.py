"""Attention at head dimensions 64 and 256 where the matrix-core kernel's lane maps can go wrong: tiles with one
token, with a token more or less than a page, windows whose ring has turned, every group size around the 16-row column
tile, walks cut into more shares than there are tiles.  The kernel dequantizes with the reference's two roundings and
keeps probabilities as fp32 numbers, so beyond the output's own fp16 rounding only fp32 sums remain."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


def _cache(D, B, H_KV, H_Q, T0, steps, seed):
    import kitty_amd
    from tests import gpu_util as u
    k, v = make_kv(B, H_KV, T0 + steps, D=D, seed=seed)
    cache = kitty_amd.KittyCache(u.cfg(H_KV, H_Q, D=D), B, 2048)
    ol = O.OracleLayer(B, 2048, H_KV, D=D, D_BOOSTED=D // 4)
    if T0:
        cache.update(u.to_dev(k[:, :, :T0]), u.to_dev(v[:, :, :T0]), 0)
        cache.quantize_prefill(0)
        ol.update(k[:, :, :T0], v[:, :, :T0])
        ol.quantize_prefill()
    for t in range(T0, T0 + steps):
        cache.update(u.to_dev(k[:, :, t:t + 1]), u.to_dev(v[:, :, t:t + 1]), 0)
        cache.quantize_decode(0)
        ol.update(k[:, :, t:t + 1], v[:, :, t:t + 1])
        ol.quantize_decode()
    return u, cache, ol


def _close(out, ref, what):
    got = out.float().cpu().numpy().astype(np.float64)
    # half a unit of the fp16 result (2^-11 of it), plus fp32 sums over a few thousand terms of size |v| <= 8
    bound = 2.0 ** -11 * np.abs(ref) + 2e-5
    assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all(), f"{what}: {np.abs(got - ref).max():.2e}"


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T0,steps", [(1, 0), (31, 2), (32, 1), (159, 0), (160, 0), (161, 0), (32 + 256, 129), (32 + 384 + 127, 3), (40, 200)])
@pytest.mark.parametrize("G", [1, 5, 16])
def test_decode(D, T0, steps, G):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    B, H_KV = 2, 1
    u, cache, ol = _cache(D, B, H_KV, G, T0, steps, seed=T0 + steps + G)
    q = np.random.default_rng(T0 + G).standard_normal((B, G, 1, D)).astype(np.float16)
    ref = O.decode_attention(ol, q, D ** -0.5, reference_rounding=False, dequant="two")
    for splits in (None, 1, 2, 7):
        out, _ = kitty_attention_forward(u.module(H_KV, G), u.to_dev(q), cache.kv_cache[0], D ** -0.5, num_splits=splits)
        _close(out, ref, f"D={D} T0={T0}+{steps} G={G} splits={splits}")


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T0,Tq,G", [(0, 1, 1), (0, 130, 3), (33, 129, 16), (32 + 128 + 5, 64, 4), (32 + 640 + 100, 17, 5)])
def test_chunk(D, T0, Tq, G, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import _lib
    from kitty_amd.kvcache.kernels import kitty_attention as A
    B, H_KV = 1, 2
    u, cache, ol = _cache(D, B, H_KV, H_KV * G, T0, 0, seed=T0 + Tq)
    k, v = make_kv(B, H_KV, Tq, D=D, seed=Tq)
    q = np.random.default_rng(Tq).standard_normal((B, H_KV * G, Tq, D)).astype(np.float16)
    ref = O.chunk_attention(ol, q, k, v, D ** -0.5, dequant="two")
    for s in (1, 3, 20):
        monkeypatch.setattr(A, "_chunk_split_plan",
                            lambda *a, s=s: (s, _lib.lib().kitty_prefill_attn_workspace_bytes(B, H_KV * G, D, Tq, s)))
        out, _ = A.kitty_prefill_attention(u.module(H_KV, H_KV * G), u.to_dev(q), u.to_dev(k), u.to_dev(v), cache.kv_cache[0],
                                           D ** -0.5)
        _close(out, ref, f"D={D} T0={T0} Tq={Tq} G={G} shares={s}")
