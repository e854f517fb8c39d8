"""The simulator after an exception inside update: nothing of a failed prompt stays, and a step's quantizations that did not run are
still there for the next call."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T = 32 + 2 * 128                    # the first step completes a block: its keys and a token's values wait for the next step


def _steps():
    g = torch.Generator(device="cuda").manual_seed(2)
    return [torch.randn(2, 1, 2, n, 128, generator=g, device="cuda").half() for n in [T] + [1] * 3]


def _stock(sim, post):
    c = sim.KittyKVCache(sim.KittyKVCacheConfig(promote_ratio=0.25, PostQuant=post), max_length=T + 3)
    for k, v in _steps():
        c.update(k, v, 0)
    c.flush_pending()
    return c


def _boom(*a, **kw):
    raise RuntimeError("boom")


def _same(a, b):
    return all(torch.equal(x[0].view(torch.int16), y[0].view(torch.int16)) for x, y in ((a.key_cache, b.key_cache), (a.value_cache, b.value_cache)))


@pytest.mark.parametrize("where", ["_quant_k_ranked", "_values_from", "_append_step"])
def test_update_again(where, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    c = sim.KittyKVCache(sim.KittyKVCacheConfig(promote_ratio=0.25), max_length=T + 3)
    for i, (k, v) in enumerate(_steps()):
        with monkeypatch.context() as m:
            m.setattr(sim.KittyKVCache, where, _boom)
            if (where == "_append_step") == (i > 0):
                with pytest.raises(RuntimeError, match="boom"):
                    c.update(k, v, 0)
                assert len(c.key_cache) == len(c.value_cache) == len(c._len) == len(c._pending) == (1 if i else 0)
        c.update(k, v, 0)
    c.flush_pending()
    assert _same(c, _stock(sim, True))


def test_waiting_quantizations_stay(monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    c = sim.KittyKVCache(sim.KittyKVCacheConfig(promote_ratio=0.25), max_length=T + 3)
    steps = _steps()
    for k, v in steps[:2]:
        c.update(k, v, 0)
    waiting = list(c._pending[0])
    assert [j[0] for j in waiting] == ["k", "v"]
    with monkeypatch.context() as m:
        m.setattr(sim, "build_promote_mask", _boom)
        with pytest.raises(RuntimeError, match="boom"):
            c.update(*steps[2], 0)
    assert c._pending[0] == waiting and c.get_seq_length() == T + 1
    for k, v in steps[2:]:
        c.update(k, v, 0)
    c.flush_pending()
    assert _same(c, _stock(sim, True))
