"""Where something else than autograd's backward follows the tensor operations, or the tensors are not on the current
device, the calls that had become single launches stay tensor operations."""
import types

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from kitty_amd import _lib


def test_launchable(monkeypatch):
    dev = torch.device("cuda", 0)
    monkeypatch.setattr(_lib, "_current_device", lambda: 0)
    assert _lib.launchable(dev) and _lib.launchable(torch.device("cuda"))
    with fwAD.dual_level():
        assert not _lib.launchable(dev)
    seen = []

    def f(x):
        seen.append(_lib.launchable(dev))
        return x + 1
    torch.jit.trace(f, torch.zeros(2), check_trace=False)
    assert seen == [False] and _lib.launchable(dev)
    monkeypatch.setattr(_lib, "_current_device", lambda: 1)
    assert not _lib.launchable(dev) and _lib.launchable(torch.device("cuda", 1))


@pytest.mark.parametrize("call", ["update", "append", "pack"])
def test_calls_stay_tensor_operations(call, monkeypatch):
    """As on a GPU, with the library's launches made an error."""
    from kitty_amd import KittyCache
    from kitty_amd.kvcache import kitty as module
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=128, num_key_value_heads=2, num_attention_heads=2, hidden_size=256)
    c = KittyCache(cfg, 2, 512, device="cpu")
    L = c.kv_cache[0]
    monkeypatch.setattr(type(L), "on_hip", True)
    monkeypatch.setattr(module._lib, "lib", lambda: pytest.fail("a kernel was launched"))
    monkeypatch.setattr(_lib, "_current_device", lambda: 0)
    T = 1 if call == "update" else 20
    x = torch.ones(2, 2, T, 128).half()
    if call != "pack":
        L.Sink_Count, L.Q_Buffer_Count_K, L.Local_Count_V = 32, 5, 5
    with fwAD.dual_level():
        if call == "append":
            c.append(x, x, 0)
        else:
            c.update(x, x, 0)
        if call == "pack":
            c.quantize_prefill(0)
    rows = L.Sink_Buffer_K[:, :, :20] if call == "pack" else L.Q_Buffer_K[:, :, 5:5 + T]
    assert bool((rows == 1).all())


def test_stream_without_the_private_name(monkeypatch):
    monkeypatch.setattr(_lib, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=77))
    assert _lib.current_stream_ptr(torch.device("cuda", 0)) == 77
