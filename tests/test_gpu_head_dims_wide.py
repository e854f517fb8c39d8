"""Decode attention at head dimensions 64 and 256 over pages with scales out of the range of the short dequantization, which end a
wavefront's own walk: none, a few early and late in walks of many pages per wavefront, and all pages of a walk."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H_Q", [(64, 4), (64, 12), (256, 4), (256, 12)])
@pytest.mark.parametrize("pages,wide", [(300, (1, 5, 6, 247, 250, 251, 252, 253, 255, 256, 270, 299)), (300, ()), (150, range(150))])
def test_wide_pages(D, H_Q, pages, wide):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    from tests import gpu_util as u
    T = 32 + 128 * pages + 128 + 40
    k, v = make_kv(1, 2, T, D=D, seed=pages + D)
    q = np.random.default_rng(D).standard_normal((1, H_Q, 1, D)).astype(np.float16)
    q[..., 3] = 0                                        # a channel that the queries do not look at
    for i, page in enumerate(wide):
        at = 32 + 128 * page + 17
        if i % 2 or len(wide) == pages:
            k[0, 0, at, 3], k[0, 0, at + 1, 3] = 600, -600
        else:
            v[0, 0, at, 5], v[0, 0, at, 6] = 300, -300
    cache = kitty_amd.KittyCache(u.cfg(2, H_Q, D=D), 1, T + 128)
    cache.update(u.to_dev(k), u.to_dev(v), 0)
    cache.quantize_prefill(0)
    ol = O.OracleLayer(1, T + 128, 2, D=D, D_BOOSTED=D // 4)
    ol.update(k, v)
    ol.quantize_prefill()
    L = cache.kv_cache[0]
    assert u.layer_bytes_equal(L, ol) == [] and L.PageCount_V == pages
    scale = L.KeyCache_metadata[L.PageTable_K[0, :pages], 0, :, 0].abs().amax(-1).maximum(
        L.ValueCache_metadata[L.PageTable_V[0, :pages], 0, :, 0].abs().amax(-1))
    assert torch.nonzero(scale >= 64).flatten().tolist() == sorted(wide)
    ref = O.decode_attention(ol, q, D ** -0.5, reference_rounding=False, dequant="two")
    # half a unit of the fp16 result, plus fp32 sums over terms of size |v| <= 8, or 300 in a token of small probability
    bound = 2.0 ** -11 * np.abs(ref) + 2e-5 * (10 if 0 < len(wide) < pages else 1)
    for splits in (1, 2, 7, None):
        out, _ = kitty_attention_forward(u.module(2, H_Q), u.to_dev(q), L, D ** -0.5, num_splits=splits)
        got = out.float().cpu().numpy().astype(np.float64)
        assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all(), (splits, np.abs(got - ref).max())
