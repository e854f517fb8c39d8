"""Layers and calls outside what the append and packing kernels are built for keep the tensor copies."""
import types

import pytest
import torch


def _cache(D, device, rows=2):
    from kitty_amd import KittyCache
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=D, num_key_value_heads=2, num_attention_heads=2, hidden_size=2 * D)
    return KittyCache(cfg, rows, 512, device=device)


@pytest.mark.parametrize("D", [96, 128])
def test_layers_know_whether_the_kernels_serve_them(D):
    assert _cache(D, "cpu").kv_cache[0].on_hip is False


@pytest.mark.gpu
def test_other_head_dims_and_broadcast_rows_still_append():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    for D, heads in ((96, 2), (128, 1)):            # a head dimension without kernels; one head for all, as a slice assignment takes it
        gpu, cpu = _cache(D, "cuda"), _cache(D, "cpu")
        assert gpu.kv_cache[0].on_hip is (D == 128)
        k, v = torch.randn(2, 2, 100, D).half(), torch.randn(2, 2, 100, D).half()
        for c, dev in ((gpu, "cuda"), (cpu, "cpu")):
            c.update(k.to(dev), v.to(dev), 0)
        gpu.quantize_prefill(0)
        cpu.quantize_prefill(0)
        for s in range(3):
            kn, vn = torch.randn(2, heads, 1, D).half(), torch.randn(2, heads, 1, D).half()
            assert gpu.update(kn.cuda(), vn.cuda(), 0) is False and cpu.update(kn, vn, 0) is False
        a, b = gpu.kv_cache[0], cpu.kv_cache[0]
        assert a.counts() == b.counts()
        for n in ("Sink_Buffer_K", "Sink_Buffer_V", "Q_Buffer_K", "Q_Buffer_V", "Local_Buffer_V"):
            assert torch.equal(getattr(a, n).cpu(), getattr(b, n)), (D, n)
