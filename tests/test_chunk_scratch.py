"""The scratch of a chunk's shares is bounded, whatever its shape (the rule needs no GPU)."""
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
