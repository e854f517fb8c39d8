"""A layer's descriptor follows its tensors: one that was replaced, or whose storage was moved, is read and written
where it is now."""
import types

import pytest
import torch

NAMES = dict(KeyCache="key_cache", KeyCache_metadata="key_meta", ValueCache="value_cache", ValueCache_metadata="value_meta",
             PageTable_K="page_table_k", PageTable_V="page_table_v", Sink_Buffer_K="sink_k", Sink_Buffer_V="sink_v",
             Q_Buffer_K="qbuf_k", Q_Buffer_V="qbuf_v", Local_Buffer_V="local_v", status="status")


def _cache(device):
    from kitty_amd import KittyCache
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=128, num_key_value_heads=2, num_attention_heads=2, hidden_size=256)
    return KittyCache(cfg, 2, 512, device=device)


def _holds(d, L):
    for n, f in NAMES.items():
        assert getattr(d, f) == getattr(L, n).data_ptr(), n
    assert list(d.counts) == L.counts()


@pytest.mark.parametrize("name", sorted(NAMES))
def test_descriptor_follows_a_replaced_tensor(name):
    L = _cache("cpu").kv_cache[0]
    first = L.descriptor()
    _holds(first, L)
    assert L.descriptor() is first
    setattr(L, name, getattr(L, name).clone())
    _holds(L.descriptor(), L)


def test_descriptor_follows_moved_storage():
    L = _cache("cpu").kv_cache[0]
    L.descriptor()
    kept = []                                            # keeps the old storage, so that the new one lies elsewhere
    for n in NAMES:
        t = getattr(L, n)
        kept.append(t.data)
        t.data = t.data.clone()
        assert t.data_ptr() != kept[-1].data_ptr()
    _holds(L.descriptor(), L)


def test_tensors_on_different_devices_are_refused():
    L = _cache("cpu").kv_cache[0]
    L.descriptor()
    L.Q_Buffer_K = L.Q_Buffer_K.to("meta")
    with pytest.raises(ValueError, match="different devices"):
        L.descriptor()


@pytest.mark.gpu
def test_tensors_replaced_after_the_prompt_are_the_ones_that_decode_uses():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    mod = types.SimpleNamespace(num_attention_heads=2, num_key_value_heads=2)
    caches = [_cache("cuda"), _cache("cuda")]
    gen = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda", dtype=torch.float16)
    k, v = rnd(2, 2, 400, 128), rnd(2, 2, 400, 128)
    for c in caches:
        c.update(k, v, 0)
        c.quantize_prefill(0)
    L, kept = caches[1].kv_cache[0], []
    for n in NAMES:
        kept.append(getattr(L, n))
        setattr(L, n, kept[-1].clone())
    olds = [t.clone() for t in kept]
    k, v, q = rnd(2, 2, 1, 128), rnd(2, 2, 1, 128), rnd(2, 2, 1, 128)
    outs = []
    for c in caches:
        assert c.update(k, v, 0) is False
        outs.append(kitty_attention_forward(mod, q, c.kv_cache[0], 128 ** -0.5)[0])
    assert torch.equal(*outs)
    for n, a, b in zip(NAMES, kept, olds):
        assert torch.equal(a, b), n                                                    # nothing was written to the old ones
        assert torch.equal(getattr(L, n), getattr(caches[0].kv_cache[0], n)), n
