"""The simulator's launches that take in the top-k, the mask and the copies against tensor operations: the same bits, for
scores full of ties, NaN and infinities, in both layouts of the source, across decode steps that flush a block."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _record(sim, monkeypatch):
    """What _quant_k_ranked (with a source, in place) and _append_step return: True, they launched; False, tensor operations follow."""
    taken = {"prompt": [], "block": [], "step": []}
    ranked, step = sim.KittyKVCache._quant_k_ranked, sim.KittyKVCache._append_step

    def record_ranked(self, K, lo, hi, src):
        taken["block" if src is None else "prompt"].append(ranked(self, K, lo, hi, src))
        return taken["block" if src is None else "prompt"][-1]

    def record_step(self, *a):
        taken["step"].append(step(self, *a))
        return taken["step"][-1]

    monkeypatch.setattr(sim.KittyKVCache, "_quant_k_ranked", record_ranked)
    monkeypatch.setattr(sim.KittyKVCache, "_append_step", record_step)
    return taken


def _data(L, kind, layout, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(2, L, 3, 128, generator=g)
    if kind == "ties":
        x = (x * 2).round().clamp(-2, 2)
        x[:, :, 1] = 1.0                                     # every channel of a head alike
    x = x.half().transpose(1, 2)
    if kind == "special":
        x[0, 0, 40, 7] = float("nan")
        x[0, 1, 41, 9] = float("inf")
        x[1, 2, 200:, 11] = float("-inf")
    return (x.contiguous() if layout == "contiguous" else x).cuda()


@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
@pytest.mark.parametrize("layout", ["token-major", "contiguous"])
@pytest.mark.parametrize("L,group,sink,ratio,sel,post,bitdec", [
    (161, 128, 32, 0.25, 1, True, False), (288, 64, 32, 0.1, 1, False, False), (415, 32, 0, 0.5, 1, True, True),
    (700, 128, 5, 0.25, 2, False, False), (300, 64, 32, 0.0, 1, True, False), (300, 128, 32, 1.0, 1, True, False)])
def test_same_bits_as_tensor_operations(kind, layout, L, group, sink, ratio, sel, post, bitdec, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    cfg = dict(sink_length=sink, group_size=group, promote_ratio=ratio, channel_selection=sel, PostQuant=post, VCache_BitDecoding=bitdec)
    steps = 140
    k, v = _data(L, kind, layout, L), _data(L, "normal", layout, L + 1)
    new = [(_data(1, "normal", layout, 10 * s), _data(1, "normal", layout, 10 * s + 1)) for s in range(steps)]
    outs = []
    taken = _record(sim, monkeypatch)
    for fused in (True, False):
        for calls in taken.values():
            calls.clear()
        if not fused:
            monkeypatch.setattr(sim._lib, "launchable", lambda device: False)
        c = sim.KittyKVCache(sim.KittyKVCacheConfig(**cfg), max_length=L + steps)
        out = [x.clone() for x in c.update(k, v, 0)]
        for i, (kn, vn) in enumerate(new):
            last = c.update(kn, vn, 0)
            if i in (0, 1, steps - 1):
                out += [x.clone() for x in last]
        c.flush_pending()
        some = fused and 0 < ratio < 1
        assert taken["step"] == [fused] * steps and len(taken["block"]) >= 1 and set(taken["block"]) == {some}
        assert taken["prompt"] == ([some and sel == 1] if L > sink + 128 else [])
        outs.append(out + [c.key_cache[0][:, :, :L + steps], c.value_cache[0][:, :, :L + steps]])
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def test_growing_buffers(monkeypatch):
    """Without max_length the buffers double when they are full, between two steps of the fused route."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    L, steps = 161, 1030
    k, v = _data(L + steps, "normal", "token-major", 1), _data(L + steps, "normal", "token-major", 2)
    taken, outs = _record(sim, monkeypatch), []
    for fused in (True, False):
        for calls in taken.values():
            calls.clear()
        if not fused:
            monkeypatch.setattr(sim._lib, "launchable", lambda device: False)
        c = sim.KittyKVCache(sim.KittyKVCacheConfig(promote_ratio=0.25))
        c.update(k[:, :, :L], v[:, :, :L], 0)
        held = c.key_cache[0].shape[2]
        for t in range(L, L + steps):
            last = c.update(k[:, :, t:t + 1], v[:, :, t:t + 1], 0)
        assert c.key_cache[0].shape[2] == 2 * held and taken["step"] == [fused] * steps
        outs.append([x.clone() for x in last])
    for a, b in zip(*outs):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))
