"""Chunked-prefill attention with its walk over the tokens cut into shares: every number of shares against the
single walk, at the edges where a share can go wrong (more shares than tiles, a share that starts inside the
chunk so that the first rows see none of it, more body tiles per share than one load of page ids, one position)."""
import pytest
import torch

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
