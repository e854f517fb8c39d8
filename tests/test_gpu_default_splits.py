"""kitty_decode_attn with num_splits = 0 and a workspace sized by either of the two rules the header names."""
import numpy as np
import pytest
import torch

from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("T", [40, 2100, 4200])
def test_workspace_by_either_rule(D, T):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd import _lib
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    from tests import gpu_util as u
    B, H_KV, H_Q = 1, 8, 16
    cache = kitty_amd.KittyCache(u.cfg(H_KV, H_Q, D=D), B, T + 256)
    k, v = make_kv(B, H_KV, T, D=D, seed=T)
    cache.update(u.to_dev(k), u.to_dev(v), 0)
    cache.quantize_prefill(0)
    L, lib = cache.kv_cache[0], _lib.lib()
    q = u.to_dev(np.random.default_rng(T).standard_normal((B, H_Q, 1, D)).astype(np.float16))
    tiles = 1 + -(-(T - 32) // 128)
    rules = (lib.kitty_decode_attn_default_splits(B, H_KV, tiles, 0), lib.kitty_decode_attn_default_splits_d(B, H_KV, D, tiles, 0))
    assert rules[0] == rules[1] or D != 128
    for splits in rules:
        want, _ = kitty_attention_forward(u.module(H_KV, H_Q), q, L, D ** -0.5, num_splits=splits)
        ws = torch.empty(lib.kitty_decode_attn_workspace_bytes(B, H_Q, D, splits), dtype=torch.uint8, device="cuda")
        out = torch.empty_like(want)
        rc = lib.kitty_decode_attn(L.descriptor(), q.data_ptr(), B, H_Q, D ** -0.5, out.data_ptr(), ws.data_ptr(), ws.numel(), 0, 0,
                                   _lib.current_stream_ptr(q.device))
        _lib.check(rc, "kitty_decode_attn")
        assert torch.equal(out, want), splits
    least = lib.kitty_decode_attn_workspace_bytes(B, H_Q, D, min(rules))    # less than either rule asks for is refused as ever
    assert lib.kitty_decode_attn(L.descriptor(), q.data_ptr(), B, H_Q, D ** -0.5, out.data_ptr(), ws.data_ptr(), least - 1, 0, 0,
                                 _lib.current_stream_ptr(q.device)) == -5
