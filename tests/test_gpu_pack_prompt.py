"""A prompt in one launch (kitty_pack_prompt) and a chunk in two (kitty_append_chunk_host) against the tensor copies
and quantizer launches of the same methods, which serve sources the kernels cannot read as they lie: every byte of
the layer and every counter, at the lengths where a part appears, fills up or turns over."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu

NAMES = ("Sink_Buffer_K", "Sink_Buffer_V", "Q_Buffer_K", "Q_Buffer_V", "Local_Buffer_V", "KeyCache", "KeyCache_metadata",
         "ValueCache", "ValueCache_metadata", "status")


def _cache(D, H, rows, max_len):
    from kitty_amd import KittyCache
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=D, num_key_value_heads=H, num_attention_heads=H, hidden_size=H * D)
    c = KittyCache(cfg, rows, max_len)
    for n in NAMES:
        getattr(c.kv_cache[0], n).zero_()
    return c


def _odd(x):
    """The same values in rows that do not start on 16 bytes."""
    wide = x.new_zeros(*x.shape[:3], x.shape[3] + 4)
    wide[..., :x.shape[3]] = x
    return wide[..., :x.shape[3]]


def _same(a, b, what):
    a, b = a.kv_cache[0], b.kv_cache[0]
    assert a.counts() == b.counts(), what
    for n in NAMES:
        x, y = getattr(a, n), getattr(b, n)
        assert torch.equal(x, y), (what, n)


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


@pytest.mark.parametrize("D,H", [(128, 3), (64, 2), (256, 1)])
@pytest.mark.parametrize("T", [1, 31, 32, 33, 159, 160, 161, 287, 288, 289, 417, 700])
def test_prompt(D, H, T):
    g = torch.Generator().manual_seed(D + T)
    B = 2
    k = torch.randn(B, T, H, D, generator=g).half().cuda().transpose(1, 2)      # token-major, as a projection leaves it
    v = torch.randn(B, H, T, D, generator=g).half().cuda()                       # strides of its own
    fast, slow = _cache(D, H, B + 1, 1024), _cache(D, H, B + 1, 1024)
    for c, f in ((fast, lambda x: x), (slow, _odd)):
        c.kv_cache[0].PageTable_K[0, 1] = 10 ** 6                                # an id outside the cache: recorded, not written
        c.update(f(k), f(v), 0)
        c.quantize_prefill(0)
    _same(fast, slow, T)
    # other rows of a layer: what a pool of pages does when it admits a prompt into a slot
    for c, f in ((fast, lambda x: x), (slow, _odd)):
        c._store_prefill(c.kv_cache[0], f(k[:1]), f(v[:1]), 2)
    _same(fast, slow, T)


@pytest.mark.parametrize("T0", [5, 32, 100, 160, 400])
@pytest.mark.parametrize("chunks", [(1, 26, 1), (27, 128, 60), (300, 1, 127), (128, 128), (513, 40)])
def test_chunk(T0, chunks):
    D, H, B = 128, 3, 2
    g = torch.Generator().manual_seed(T0 + len(chunks))
    fast, slow = _cache(D, H, B, 2048), _cache(D, H, B, 2048)
    for n in (T0,) + chunks:
        k, v = (torch.randn(B, n, H, D, generator=g).half().cuda().transpose(1, 2) for _ in range(2))
        fast.append(k, v, 0)
        slow.append(_odd(k), _odd(v), 0)
        _same(fast, slow, (T0, chunks, n))
    k = torch.zeros(B, H, 2400, D, device="cuda", dtype=torch.float16)
    before = fast.kv_cache[0].counts()
    with pytest.raises(ValueError, match="max_length"):
        fast.append(k, k, 0)
    assert fast.kv_cache[0].counts() == before


@pytest.mark.parametrize("side,entry", [("K", 0), ("K", 2), ("V", 0), ("V", 1)])
@pytest.mark.parametrize("T0,T", [(100, 600), (40, 500), (32 + 128, 500)])
def test_chunk_records_a_page_id_outside_the_cache(side, entry, T0, T):
    """Both routes: the page is not written, everything else is, and ``check_status`` says whose page it was."""
    D, H, B = 128, 2, 2
    g = torch.Generator().manual_seed(T0 + T)
    fast, slow, whole = (_cache(D, H, B, 2048) for _ in range(3))
    rows = [tuple(torch.randn(B, n, H, D, generator=g).half().cuda().transpose(1, 2) for _ in range(2)) for n in (T0, T)]
    for c in (fast, slow):
        getattr(c.kv_cache[0], "PageTable_" + side)[1, entry] = 10 ** 6
    for c, f in ((fast, lambda x: x), (slow, _odd), (whole, lambda x: x)):
        for k, v in rows:
            c.append(f(k), f(v), 0)
    _same(fast, slow, (side, entry))
    for c in (fast, slow):
        assert c.check_status(raise_on_error=False)["bad_page_write"].tolist() == [[0, 1]]
        with pytest.raises(RuntimeError, match="bad_page_write"):
            c.check_status()
    whole.check_status()
    L, W = fast.kv_cache[0], whole.kv_cache[0]
    name = "KeyCache" if side == "K" else "ValueCache"
    assert not getattr(L, name)[L.MAX_PAGE + entry].any() and getattr(W, name)[L.MAX_PAGE + entry].any()
