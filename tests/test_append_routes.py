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


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 128, 256])
def test_layers_with_counters_set_by_hand_still_append(D):
    """``seq_counts`` assigned without ``enable_device_counters``: attention reads them, ``update`` and ``append`` go by
    the host ints, as on any layer."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    by_hand, plain = _cache(D, "cuda"), _cache(D, "cuda")
    gen = torch.Generator(device="cuda").manual_seed(D)
    rnd = lambda T: torch.randn(2, 2, T, D, generator=gen, device="cuda", dtype=torch.float16)
    a, b = by_hand.kv_cache[0], plain.kv_cache[0]
    rows = [rnd(100), rnd(100)]
    for c in (by_hand, plain):
        c.update(*rows, 0)
        c.quantize_prefill(0)
    a.seq_counts = torch.tensor([a.counts()] * 2, dtype=torch.int32, device="cuda")
    for T in (1, 1, 70, 1):
        rows = [rnd(T), rnd(T)]
        for c in (by_hand, plain):
            if T == 1:
                assert c.update(*rows, 0) is False
                c.quantize_decode(0)
            else:
                c.append(*rows, 0)
    assert a.counts() == b.counts()
    for n in ("Sink_Buffer_K", "Sink_Buffer_V", "Q_Buffer_K", "Q_Buffer_V", "Local_Buffer_V", "KeyCache", "KeyCache_metadata",
              "ValueCache", "ValueCache_metadata"):
        assert torch.equal(getattr(a, n), getattr(b, n)), n


@pytest.mark.parametrize("D", [64, 128, 256])
def test_counters_set_by_hand_take_the_copies(D, monkeypatch):
    from kitty_amd.kvcache import kitty as module
    c = _cache(D, "cpu")
    L = c.kv_cache[0]
    L.Sink_Count, L.Q_Buffer_Count_K, L.Local_Count_V = 32, 5, 5
    L.seq_counts = torch.tensor([L.counts()] * 2, dtype=torch.int32)
    monkeypatch.setattr(type(L), "on_hip", True)                       # as on a GPU, but a launch is an error
    monkeypatch.setattr(module._lib, "lib", lambda: pytest.fail("a kernel was launched"))
    x = torch.ones(2, 2, 1, D).half()
    assert c.update(x, x, 0) is False and L.Q_Buffer_Count_K == 6 and bool((L.Q_Buffer_K[:, :, 5] == 1).all())
    x = torch.full((2, 2, 3, D), 2.0).half()
    c.append(x, x, 0)
    assert L.Q_Buffer_Count_K == 9 and bool((L.Q_Buffer_K[:, :, 6:9] == 2).all()) and bool((L.Local_Buffer_V[:, :, 6:9] == 2).all())


def _odd_layer(device, S, max_len):
    from kitty_amd.kvcache.utils_kv_per_layer import KVCache_Layer
    c = _cache(128, device)
    c.kv_cache[0] = KVCache_Layer(2, max_len, 2, 128, 32, 2, 4, 128, S, device=device)
    return c


@pytest.mark.gpu
@pytest.mark.parametrize("S,max_len,steps", [(0, 512, (300,)), (0, 512, (300, 40)), (32, 0, (50, 1, 30))])
def test_layers_without_a_sink_or_without_pages_still_take_tokens(S, max_len, steps):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    c = _odd_layer("cuda", S, max_len)
    L = c.kv_cache[0]
    gen = torch.Generator(device="cuda").manual_seed(5)
    K = torch.randn(2, 2, sum(steps), 128, generator=gen, device="cuda", dtype=torch.float16)
    V = torch.randn(2, 2, sum(steps), 128, generator=gen, device="cuda", dtype=torch.float16)
    c.update(K[:, :, :steps[0]], V[:, :, :steps[0]], 0)
    c.quantize_prefill(0)
    t = steps[0]
    for n in steps[1:]:
        if n == 1:
            assert c.update(K[:, :, t:t + 1], V[:, :, t:t + 1], 0) is False
        else:
            c.append(K[:, :, t:t + n], V[:, :, t:t + n], 0)
        t += n
    assert L.get_total_length() == t and L.PageCount_K == (t - S) // 128
    rk = L.Q_Buffer_Count_K
    assert torch.equal(L.Q_Buffer_K[:, :, :rk], K[:, :, t - rk:t]) and torch.equal(L.Sink_Buffer_K, K[:, :, :S])


@pytest.mark.parametrize("S,max_len", [(0, 512), (32, 0)])
def test_layers_without_a_sink_or_without_pages_are_not_for_the_kernels(S, max_len, monkeypatch):
    L = _odd_layer("cpu", S, max_len).kv_cache[0]
    monkeypatch.setattr(type(L), "_KeyCache", types.SimpleNamespace(is_cuda=True), raising=False)
    del L.__dict__["_KeyCache"]
    assert L.on_hip is False
    L._kernel_shape = True
    assert L.on_hip is True
