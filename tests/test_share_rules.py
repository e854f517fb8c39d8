"""How many shares a walk over the tokens is cut into (the rules need no GPU): the scratch of a chunk's shares is bounded,
and no share is empty."""
import itertools

import pytest


@pytest.mark.parametrize("D", [64, 128, 256])
def test_scratch_is_bounded(D):
    from kitty_amd import _lib
    lib = _lib.lib()
    cut = 0
    for B, (H_Q, H_KV), T_q, tiles in itertools.product(
            (1, 2, 3, 4, 8, 16, 64), ((64, 8), (40, 8), (32, 8), (32, 2), (16, 16), (8, 1)),
            (1, 16, 130, 576, 1116, 1900, 2050, 3500, 16384), (1, 20, 96, 257, 1024)):
        s = lib.kitty_prefill_attn_default_splits(B, H_Q, H_KV, D, T_q, tiles)
        assert s >= 1 and (s == 1 or lib.kitty_prefill_attn_workspace_bytes(B, H_Q, D, T_q, s) <= 128 << 20), (B, H_Q, H_KV, T_q, tiles, s)
        cut += s > 1
    assert cut > 100                                       # the rule still cuts walks


def test_no_share_is_empty_at_head_dim_256():
    """Equal shares of ceil(tiles / shares) tiles: the default counts leave none of them without a tile."""
    from kitty_amd import _lib
    lib = _lib.lib()
    for B, H_KV, tiles in itertools.product((1, 2, 3, 4, 9, 40), (1, 2, 8), (1, 2, 5, 17, 33, 65, 71, 72, 200, 236, 1025)):
        s = lib.kitty_decode_attn_default_splits_d(B, H_KV, 256, tiles, 0)
        assert (s - 1) * -(-tiles // s) < tiles, (B, H_KV, tiles, s)
        for T_q in (3, 16, 200, 900):
            n = tiles + -(-T_q // 128)
            s = lib.kitty_prefill_attn_default_splits(B, 4 * H_KV, H_KV, 256, T_q, tiles)
            assert (s - 1) * -(-n // s) < n, (B, H_KV, tiles, T_q, s)
