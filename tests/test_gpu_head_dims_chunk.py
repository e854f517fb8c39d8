"""A chunk in two launches at head dimensions 64 and 256 (kitty_append_chunk_host_d) against the tensor copies and quantizer
launches that serve sources the kernels cannot read as they lie: every byte of the layer and every counter, where a sink, a
Q-buffer, the ring or a page begins, fills up or turns over.  kitty_append_chunk_host itself still takes 128 alone."""
import pytest
import torch

from tests.test_gpu_pack_prompt import _cache, _odd, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,H", [(64, 3), (256, 2)])
@pytest.mark.parametrize("T0", [5, 32, 160, 400])
@pytest.mark.parametrize("chunks", [(1, 26, 1), (27, 128, 60), (300, 1, 127), (513, 40)])
def test_chunk(D, H, T0, chunks):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import _lib
    B = 2
    g = torch.Generator().manual_seed(T0 + len(chunks) + D)
    fast, slow = _cache(D, H, B, 2048), _cache(D, H, B, 2048)
    for c in (fast, slow):
        c.kv_cache[0].PageTable_V[1, 1] = 10 ** 6                                # an id outside the cache: recorded, not written
    for n in (T0,) + chunks:
        k, v = (torch.randn(B, n, H, D, generator=g).half().cuda().transpose(1, 2) for _ in range(2))
        fast.append(k, v, 0)
        slow.append(_odd(k), _odd(v), 0)
        _same(fast, slow, (T0, chunks, n))
    L = fast.kv_cache[0]
    st = [2 * s for s in k.stride()[:3]]
    rc = _lib.lib().kitty_append_chunk_host(L.descriptor(), k.data_ptr(), v.data_ptr(), *st, B, 1, 0)
    assert rc < 0 and b"head_dim 128" in _lib.lib().kitty_last_error()
