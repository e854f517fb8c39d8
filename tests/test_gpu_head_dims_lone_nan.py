"""Decode at head dimensions 64 and 256: a row that meets a NaN logit is 0 also where a share of the walk met nothing else - a tail tile of
one token, a sink of NaN keys, a page with a NaN scale - with few tiles and many, in the default number of shares and in others.  Every
other row keeps its bits."""
import numpy as np
import pytest
import torch

from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T", [32 + 1, 32 + 128 + 1, 32 + 128 * 5 + 1, 32 + 128 * 66 + 1])   # (the last: more tiles than compute units)
@pytest.mark.parametrize("splits", [None, 1, 5, 20])
@pytest.mark.parametrize("H_Q", [4, 16])
def test_decode(D, T, splits, H_Q):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    from tests import gpu_util as u
    k, v = make_kv(2, 2, T, D=D, seed=T)
    cache = kitty_amd.KittyCache(u.cfg(2, H_Q, D=D), 2, T + 128)
    cache.update(u.to_dev(k), u.to_dev(v), 0)
    cache.quantize_prefill(0)
    L, G = cache.kv_cache[0], H_Q // 2
    q = u.to_dev(np.random.default_rng(T).standard_normal((2, H_Q, 1, D)).astype(np.float16))

    def run():
        return kitty_attention_forward(u.module(2, H_Q), q, L, D ** -0.5, num_splits=splits)[0].cpu()

    clean = run()
    assert torch.isfinite(clean).all() and (clean != 0).any(-1).all()
    page = int(L.PageTable_K[1, L.PageCount_K - 1]) if L.PageCount_K else -1
    places = [("tail", L.Q_Buffer_K[1, 0, 0]), ("sink", L.Sink_Buffer_K[1, 0])] + ([("page", L.KeyCache_metadata[page, 0, 0])] if page >= 0 else [])
    for what, place in places:
        kept = place.clone()
        place.fill_(float("nan"))
        got = run()
        place.copy_(kept)
        assert (got[1, 0, :G] == 0).all(), what
        got[1, 0, :G] = clean[1, 0, :G]
        assert torch.equal(got, clean), what
