"""A layer can be copied and pickled at any time (a prompt's cache is reused that way), also after its descriptor exists."""
import copy
import pickle
import types

import pytest
import torch


def _cache(device):
    from kitty_amd import KittyCache
    cfg = types.SimpleNamespace(num_hidden_layers=2, head_dim=128, num_key_value_heads=2, num_attention_heads=2, hidden_size=256)
    return KittyCache(cfg, 1, 512, device=device)


@pytest.mark.parametrize("how", [copy.deepcopy, lambda c: pickle.loads(pickle.dumps(c))], ids=["deepcopy", "pickle"])
def test_copy_after_the_descriptor_exists(how):
    c = _cache("cpu")
    for L in c.kv_cache:
        L.Q_Buffer_K.normal_()
        L.Sink_Count, L.Q_Buffer_Count_K, L.Local_Count_V = 32, 5, 5
        L.descriptor()
    d = how(c)
    for a, b in zip(c.kv_cache, d.kv_cache):
        assert a.counts() == b.counts() and torch.equal(a.Q_Buffer_K, b.Q_Buffer_K)
        b.Q_Buffer_Count_K = b.Local_Count_V = 7
        x, y = a.descriptor(), b.descriptor()
        assert y.qbuf_k == b.Q_Buffer_K.data_ptr() != x.qbuf_k == a.Q_Buffer_K.data_ptr()
        assert list(y.counts) == b.counts() and list(x.counts) == a.counts()
        assert y.qbuf_k != 0 and b.workspace(16).data_ptr() != a.workspace(16).data_ptr()


@pytest.mark.gpu
def test_a_copied_prompt_decodes_as_the_original():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    c = _cache("cuda")
    gen = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda", dtype=torch.float16)
    for l in range(2):
        c.update(rnd(1, 2, 300, 128), rnd(1, 2, 300, 128), l)
        c.quantize_prefill(l)
    d = copy.deepcopy(c)
    mod = types.SimpleNamespace(num_attention_heads=2, num_key_value_heads=2)
    for _ in range(3):
        k, v, q = rnd(1, 2, 1, 128), rnd(1, 2, 1, 128), rnd(1, 2, 1, 128)
        outs = []
        for x in (c, d):
            assert x.update(k, v, 0) is False
            outs.append(kitty_attention_forward(mod, q, x.kv_cache[0], 128 ** -0.5)[0])
            x.quantize_decode(0)
        assert torch.equal(*outs)
