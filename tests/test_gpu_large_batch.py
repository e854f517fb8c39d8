"""A batch of more sequences than a launch's grid takes: the fp16 rows of a prompt, of steps and of a chunk go in by tensor copies."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
def test_rows_of_a_large_batch(D):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import KittyCache
    B, T = 65536, 40 + 2 + 30
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=D, num_key_value_heads=1, num_attention_heads=1, hidden_size=D)
    cache = KittyCache(cfg, B, 128)
    g = torch.Generator(device="cuda").manual_seed(D)
    k, v = (torch.randn(B, 1, T, D, generator=g, device="cuda", dtype=torch.float16) for _ in range(2))
    cache.update(k[:, :, :40], v[:, :, :40], 0)
    cache.quantize_prefill(0)
    for t in (40, 41):
        assert cache.update(k[:, :, t:t + 1], v[:, :, t:t + 1], 0) is False
        cache.quantize_decode(0)
    cache.append(k[:, :, 42:], v[:, :, 42:], 0)
    L = cache.kv_cache[0]
    assert L.counts()[:7] == [32, 0, T - 32, 0, 0, T - 32, 0]
    assert torch.equal(L.Sink_Buffer_K, k[:, :, :32]) and torch.equal(L.Sink_Buffer_V, v[:, :, :32])
    assert torch.equal(L.Q_Buffer_K[:, :, :T - 32], k[:, :, 32:]) and torch.equal(L.Local_Buffer_V[:, :, :T - 32], v[:, :, 32:])
