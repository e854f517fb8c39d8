"""Decode attention at head dimensions 64 and 256 over more tiles than compute units, on either side of the line between the
two decode kernels (test_gpu_head_dims_few has more on the far side): whole pages beside tiles with fp16 rows.  Group sizes on either side of the limit for parts in columns, walks cut into few and many splits (a
wavefront with none, one and several pages), scales and zeros out of the range of the short dequantization, a high plane
of another size.  Beyond the output's own fp16 rounding only fp32 sums remain (test_gpu_head_dims_edges)."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


def _layer(D, B, H_KV, H_Q, k, v, boosted=None):
    import kitty_amd
    from kitty_amd.kvcache.utils_kv_per_layer import KVCache_Layer
    from tests import gpu_util as u
    T = k.shape[2]
    cache = kitty_amd.KittyCache(u.cfg(H_KV, H_Q, D=D), B, T + 256)
    boosted = D // 4 if boosted is None else boosted
    if boosted != D // 4:
        cache.kv_cache[0] = KVCache_Layer(MAX_BS=B, MAX_LEN=T + 256, H_KV=H_KV, D=D, D_BOOSTED=boosted, LOW_BIT=2, HIGH_BIT=4,
                                          PAGE_SIZE=128, S=32, device="cuda")
    ol = O.OracleLayer(B, T + 256, H_KV, D=D, D_BOOSTED=boosted)
    cache.update(u.to_dev(k), u.to_dev(v), 0)
    cache.quantize_prefill(0)
    ol.update(k, v)
    ol.quantize_prefill()
    assert u.layer_bytes_equal(cache.kv_cache[0], ol) == []
    return u, cache, ol


def _check(u, cache, ol, q, D, H_KV, G, splits, what, scale=1.0, rows=None):
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    ref = O.decode_attention(ol, q, D ** -0.5, reference_rounding=False, dequant="two")
    for s in splits:
        out, _ = kitty_attention_forward(u.module(H_KV, H_KV * G), u.to_dev(q), cache.kv_cache[0], D ** -0.5, num_splits=s)
        got = out.float().cpu().numpy().astype(np.float64)
        # half a unit of the fp16 result, plus fp32 sums over a few thousand terms of size |v| <= 8 scale
        bound = 2.0 ** -11 * np.abs(ref) + 2e-5 * scale
        assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all(), f"{what} splits={s}: {np.abs(got - ref).max():.2e}"


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("G,T", [(1, 32 + 128 * 6), (4, 32 + 128 * 7 + 9), (5, 32 + 128 * 8 + 127), (6, 32 + 128 * 6 + 1), (16, 32 + 128 * 7 + 64)])
def test_pages(D, G, T):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    B, H_KV = 25, 2                                          # 50 walks of seven tiles and more
    k, v = make_kv(B, H_KV, T, D=D, seed=T + G)
    u, cache, ol = _layer(D, B, H_KV, H_KV * G, k, v)
    q = np.random.default_rng(G).standard_normal((B, H_KV * G, 1, D)).astype(np.float16)
    _check(u, cache, ol, q, D, H_KV, G, (None, 1, 2, 3, 9, 30), f"D={D} G={G} T={T}")


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("side", ["k", "v", "zero"])
def test_scales_out_of_the_short_range(D, side):
    """A few pages with a scale of 64 and more (or a zero beyond 2^13) among ordinary ones."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    B, H_KV, G, T = 25, 2, 3, 32 + 128 * 9 + 5
    k, v = make_kv(B, H_KV, T, D=D, seed=D)
    q = np.random.default_rng(5).standard_normal((B, H_KV * G, 1, D)).astype(np.float16)
    big = 1.0
    for page in (0, 2, 6):
        at = 32 + 128 * page + 17
        if side == "k":                                      # a channel that the queries do not look at
            k[::2, 0, at, 3] = 600
            k[::2, 0, at + 1, 3] = -600
            q[..., 3] = 0
        elif side == "v":
            v[::2, 1, at, 5], v[::2, 1, at, 6] = 300, -300
            big = 40.0
        else:
            v[::2, 1, at] += np.float16(-10000)
            big = 1250.0
    u, cache, ol = _layer(D, B, H_KV, H_KV * G, k, v)
    _check(u, cache, ol, q, D, H_KV, G, (None, 1, 3), f"D={D} {side}", scale=big)


@pytest.mark.parametrize("D,boosted", [(64, 0), (64, 32), (256, 0), (256, 80)])
def test_other_high_planes(D, boosted):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    B, H_KV, G, T = 25, 2, 4, 32 + 128 * 6 + 40
    k, v = make_kv(B, H_KV, T, D=D, seed=boosted)
    u, cache, ol = _layer(D, B, H_KV, H_KV * G, k, v, boosted)
    q = np.random.default_rng(6).standard_normal((B, H_KV * G, 1, D)).astype(np.float16)
    _check(u, cache, ol, q, D, H_KV, G, (None, 1, 5), f"D={D} boosted={boosted}")
