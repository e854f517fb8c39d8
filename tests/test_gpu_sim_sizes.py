"""The simulator's launches at sizes where tensor operations have no limit: an empty batch, a batch beyond the launch's grid, a buffer of more
than 2^24 tokens."""
import pytest
import torch


@pytest.mark.gpu
@pytest.mark.parametrize("B", [0, 1, 65536])
def test_steps_of_any_batch(B):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    c = sim.KittyKVCache(sim.KittyKVCacheConfig(), max_length=36)
    k, v = (torch.randn(B, 1, 35, 128, device="cuda").half() for _ in range(2))
    c.update(k[:, :, :33], v[:, :, :33], 0)
    for t in (33, 34):
        K, V = c.update(k[:, :, t:t + 1], v[:, :, t:t + 1], 0)
    assert torch.equal(K, k) and torch.equal(V, v)      # (nothing past the sink's 32 tokens and the buffer's 128)


def test_ranked_launch_in_a_long_buffer():
    from kitty_amd import _lib
    lib = _lib.lib()

    def topk(src, T):
        return lib.kitty_fake_quant_topk(src, 256 * T, 256 * T, 256, 16, 256 * T, 256 * T, 256, 0, 1, T, 128, 0, 128, 128, 2, 16, 32, 4, None)

    assert topk(None, 1 << 25) == 0 and topk(16, 1 << 24) == 0      # (an empty batch: nothing is launched)
    assert topk(16, 1 << 25) == -3
