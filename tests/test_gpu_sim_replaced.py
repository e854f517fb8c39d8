"""The simulator with one of its quantizers replaced: what replaces it is called for every range that the stock one quantizes, prompt
and decode steps, and the bits are the same."""
import pytest
import torch

pytestmark = pytest.mark.gpu

STEPS = 140


def _run(sim, how, post, monkeypatch):
    calls = []
    cls = sim.KittyKVCache

    def recording(name, inner, bound):
        def f(*a, **kw):
            calls.append((name,) + tuple(x for x in a[bound:] if not isinstance(x, torch.Tensor)))
            return inner(*a, **kw)
        return f

    if how == "subclass":
        cls = type("Mine", (sim.KittyKVCache,), {n: recording(n, getattr(sim.KittyKVCache, n), 1)
                                                 for n in ("_quant_k", "_quant_v", "flush_pending")})
    elif how == "class":
        for n in ("_quant_k", "_quant_v"):
            monkeypatch.setattr(cls, n, recording(n, getattr(cls, n), 1))
    elif how == "function":
        monkeypatch.setattr(sim, "fake_quant_tokens_", recording("fake_quant_tokens_", sim.fake_quant_tokens_, 0))
    elif how == "mask":
        monkeypatch.setattr(sim, "build_promote_mask", recording("build_promote_mask", sim.build_promote_mask, 0))
    c = cls(sim.KittyKVCacheConfig(promote_ratio=0.25, PostQuant=post), max_length=420 + STEPS)
    if how == "object":
        for n in ("_quant_k", "_quant_v"):
            setattr(c, n, recording(n, getattr(c, n), 0))
    g = torch.Generator(device="cuda").manual_seed(1)
    for T in [420] + [1] * STEPS:
        x = torch.randn(2, 2, 3, T, 128, generator=g, device="cuda").half()
        c.update(x[0], x[1], 0)
    c.flush_pending()
    return calls, [c.key_cache[0], c.value_cache[0]]


@pytest.mark.parametrize("post", [True, False])
@pytest.mark.parametrize("how", ["subclass", "class", "object", "function", "mask"])
def test_replacement_is_called(how, post, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    with monkeypatch.context() as m:
        calls, got = _run(sim, how, post, m)
    with monkeypatch.context() as m:
        m.setattr(sim._lib, "launchable", lambda device: False)
        want_calls, want = _run(sim, how, post, m)
    assert len(want_calls) > (1 if how == "mask" else STEPS) and calls == want_calls
    with monkeypatch.context() as m:
        stock = _run(sim, None, post, m)[1]
    for a, b, c in zip(got, want, stock):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and torch.equal(a.view(torch.int16), c.view(torch.int16))
