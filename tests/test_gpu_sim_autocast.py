"""The simulator's cache filled under autocast, which computes a variance's scores in fp32: the bits of the tensor route."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("selection", [1, 2])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bits_under_autocast(selection, dtype, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    g = torch.Generator(device="cuda").manual_seed(3)
    gain = 1 + 9 * (torch.rand(1, 1, 2, 1, 128, generator=g, device="cuda") < 0.1).half()
    x = [torch.randn(2, 2, 2, n, 128, generator=g, device="cuda").half() * gain for n in [32 + 3 * 128 + 100] + [1] * 70]
    outs = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(sim._lib, "launchable", lambda device: False)
        c = sim.KittyKVCache(sim.KittyKVCacheConfig(promote_ratio=0.25, channel_selection=selection), max_length=32 + 3 * 128 + 170)
        with torch.autocast("cuda", dtype=dtype):
            for k, v in x:
                c.update(k, v, 0)
            c.flush_pending()
        outs.append((c.key_cache[0], c.value_cache[0]))
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
