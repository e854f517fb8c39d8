"""Chunked-prefill attention with its walk over the tokens cut into shares: every number of shares against the
single walk and the oracle, at the edges where a share can go wrong (more shares than tiles, a share that starts inside the
chunk so that the first rows see none of it, more body tiles per share than one load of page ids, one position)."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T0,Tq,G", [(0, 300, 4), (7, 1, 4), (33, 130, 2), (32 + 128 * 5 + 90, 200, 4), (32 + 128 * 150, 65, 16),
                                     (32 + 128 * 140 + 5, 3, 1), (500, 700, 12)])
def test_shares_agree_with_the_single_walk(T0, Tq, G, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd import _lib
    from kitty_amd.kvcache.kernels import kitty_attention as A
    from tests import gpu_util as u
    B, H_KV, D = 2, 2, 128
    cache = kitty_amd.KittyCache(u.cfg(H_KV, H_KV * G), B, T0 + Tq + 256)
    k, v = make_kv(B, H_KV, T0 + Tq, seed=T0 + Tq)
    if T0:
        cache.update(u.to_dev(k[:, :, :T0]), u.to_dev(v[:, :, :T0]), 0)
        cache.quantize_prefill(0)
    q = torch.randn(B, H_KV * G, Tq, D, generator=torch.Generator().manual_seed(T0)).half().cuda()
    outs = []
    for s in (1, 2, 3, 8, 40):
        monkeypatch.setattr(A, "_chunk_split_plan",
                            lambda *a, s=s: (s, _lib.lib().kitty_prefill_attn_workspace_bytes(B, H_KV * G, D, Tq, s)))
        out, _ = A.kitty_prefill_attention(u.module(H_KV, H_KV * G), q, u.to_dev(k[:, :, T0:]), u.to_dev(v[:, :, T0:]),
                                           cache.kv_cache[0], D ** -0.5)
        outs.append(out.float())
    # probabilities carry fp16's half unit (2^-11) in both runs, against different running maxima; the output another
    bound = 2 ** -10 * float(abs(v).max()) + 2 ** -10 * float(outs[0].abs().max())
    for s, o in zip((2, 3, 8, 40), outs[1:]):
        assert (o - outs[0]).abs().max().item() <= bound, s


@pytest.mark.parametrize("B,H_Q,H_KV,T_q,tiles", [(1, 32, 8, 200, 96), (4, 32, 8, 2048, 241), (1, 8, 8, 1, 1), (8, 16, 1, 4096, 600)])
def test_default_shares(B, H_Q, H_KV, T_q, tiles):
    """A launch that fills the device alone is not cut; one that does not is; never more than two tiles a share allow."""
    from kitty_amd import _lib
    s = _lib.lib().kitty_prefill_attn_default_splits(B, H_Q, H_KV, 128, T_q, tiles)
    assert 1 <= s <= max(1, (tiles + -(-T_q // 128)) // 2)
    if (B, T_q) == (1, 200):
        assert s > 4
    if B * T_q * H_Q // 256 >= 1024:
        assert s == 1


def _forced(monkeypatch, A, B, H_Q, T_q, s):
    from kitty_amd import _lib
    monkeypatch.setattr(A, "_chunk_split_plan",
                        lambda *a: (s, _lib.lib().kitty_prefill_attn_workspace_bytes(B, H_Q, 128, T_q, s)))


def _within(out, ref, values, what):
    """fp16 probabilities (half a unit, 2^-11, of each) weigh rows of at most max |value|; half a unit of the fp16 result."""
    got = out.float().cpu().numpy().astype(np.float64)
    bound = 2.0 ** -11 * max(float(np.abs(v).max()) for v in values) + 2.0 ** -11 * np.abs(ref)
    assert np.isfinite(got).all() and (np.abs(got - ref) <= bound).all(), (what, (np.abs(got - ref) / bound).max())


@pytest.mark.parametrize("T0,Tq,G", [(7, 130, 4), (32 + 128 * 5 + 90, 200, 4), (32 + 128 * 9, 65, 16), (300, 3, 1)])
def test_shares_against_the_oracle(T0, Tq, G, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd.kvcache.kernels import kitty_attention as A
    from tests import gpu_util as u
    B, H_KV = 1, 2
    cache = kitty_amd.KittyCache(u.cfg(H_KV, H_KV * G), B, 2048)
    ol = O.OracleLayer(B, 2048, H_KV)
    k, v = make_kv(B, H_KV, T0 + Tq, seed=T0 + Tq + 1)
    cache.update(u.to_dev(k[:, :, :T0]), u.to_dev(v[:, :, :T0]), 0)
    cache.quantize_prefill(0)
    ol.update(k[:, :, :T0], v[:, :, :T0])
    ol.quantize_prefill()
    kc, vc = k[:, :, T0:], v[:, :, T0:]
    q = np.random.default_rng(T0).standard_normal((B, H_KV * G, Tq, 128)).astype(np.float16)
    ref = O.chunk_attention(ol, q, kc, vc, 128 ** -0.5)
    for s in (1, 2, 3, 8, 40):
        _forced(monkeypatch, A, B, H_KV * G, Tq, s)
        out, _ = A.kitty_prefill_attention(u.module(H_KV, H_KV * G), u.to_dev(q), u.to_dev(kc), u.to_dev(vc), cache.kv_cache[0], 128 ** -0.5)
        _within(out, ref, (O.gather_dense_kv(ol, 0)[1], vc), s)


@pytest.mark.parametrize("Tq,s", [(90, 2), (90, 5), (300, 3), (1, 7), (90, 40)])
def test_shares_of_a_ragged_batch(Tq, s, monkeypatch):
    """Per-sequence counters: every sequence cuts its own walk, from less than a tile to nine of them and the chunk's."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd.kvcache.kernels import kitty_attention as A
    from tests import gpu_util as u
    H_KV, H_Q, lengths = 2, 8, (20, 32 + 128, 32 + 128 * 3 + 77, 32 + 128 * 8 + 127)
    B = len(lengths)
    cache = kitty_amd.KittyCache(u.cfg(H_KV, H_Q), B, 2048)
    L, ols, counts = cache.kv_cache[0], [], []
    for b, T in enumerate(lengths):
        k, v = make_kv(1, H_KV, T, seed=50 + b)
        ol = O.OracleLayer(1, 2048, H_KV)
        ol.update(k, v)
        ol.quantize_prefill()
        for n in ("Sink_Buffer_K", "Sink_Buffer_V", "Q_Buffer_K", "Q_Buffer_V", "Local_Buffer_V"):
            getattr(L, n)[b].copy_(u.to_dev(getattr(ol, n)[0]))
        for n in ("KeyCache", "KeyCache_metadata", "ValueCache", "ValueCache_metadata"):
            getattr(L, n)[b * L.MAX_PAGE:(b + 1) * L.MAX_PAGE].copy_(u.to_dev(getattr(ol, n)))
        ols.append(ol)
        counts.append([ol.Sink_Count, ol.PageCount_K, ol.Q_Buffer_Count_K, ol.PageCount_V, ol.Q_Buffer_Count_V, ol.Local_Count_V,
                       ol.Write_Offset_Local_V, 0])
    L.seq_counts = torch.tensor(counts, dtype=torch.int32, device="cuda")
    kc, vc = make_kv(B, H_KV, Tq, seed=60)
    q = np.random.default_rng(Tq).standard_normal((B, H_Q, Tq, 128)).astype(np.float16)
    _forced(monkeypatch, A, B, H_Q, Tq, s)
    out, _ = A.kitty_prefill_attention(u.module(H_KV, H_Q), u.to_dev(q), u.to_dev(kc), u.to_dev(vc), L, 128 ** -0.5)
    for b in range(B):
        ref = O.chunk_attention(ols[b], q[b:b + 1], kc[b:b + 1], vc[b:b + 1], 128 ** -0.5)
        _within(out[b:b + 1], ref, (O.gather_dense_kv(ols[b], 0)[1], vc), (s, b))
