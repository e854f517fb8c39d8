"""At head dimensions 64 and 256 probabilities enter the product with the values as fp32 numbers (in three fp16
operands).  One token per channel, so that a channel of a partial output is a probability."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("step", [0.5311, 0.7311, 0.9173])
def test_partials_hold_fp32_probabilities(D, packed, step):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd import _lib
    from tests import gpu_util as u
    H_Q, T = 4, 32 + (256 if packed else 0)                 # 256 body tokens: two packed K pages, one packed V page
    cache = kitty_amd.KittyCache(u.cfg(1, H_Q, D=D), 1, 1024)
    L, lib = cache.kv_cache[0], _lib.lib()
    k, v = np.zeros((1, 1, T, D), np.float16), np.zeros((1, 1, T, D), np.float16)
    k[0, 0, :, 0] = -30
    k[0, 0, 0, 0] = 0                                       # the row's largest logit, with values of 0
    # the tokens that the first token's wavefront owns: 8 i and 8 i + 1 of a tile
    own = [8 * i + e for i in range(1, 8 if packed else 4) for e in (0, 1)]
    at = [32 + t if packed else t for t in own]
    levels = np.linspace(1, 15, len(own)).astype(int)       # -30 + 2 (15 - level): sixteen levels, which four bits hold exactly
    for i, (t, n) in enumerate(zip(at, levels)):
        k[0, 0, t, 0] = -2 * n
        v[0, 0, t, i] = 3                                   # codes 0 and 3 at scale 1
    if packed:
        k[0, 0, 33, 0] = 0                                  # so that the page's grid is the one above
    cache.update(u.to_dev(k), u.to_dev(v), 0)
    cache.quantize_prefill(0)
    assert (L.PageCount_K, L.PageCount_V) == ((2, 1) if packed else (0, 0))
    q = torch.zeros(1, H_Q, 1, D, device="cuda", dtype=torch.float16)
    q[..., 0] = 1
    scaling = np.float32(step * np.log(2))
    ws = torch.empty(lib.kitty_decode_attn_workspace_bytes(1, H_Q, D, 1), dtype=torch.uint8, device="cuda")
    rc = lib.kitty_decode_attn_split(L.descriptor(), q.data_ptr(), 1, H_Q, float(scaling), ws.data_ptr(), ws.numel(), 1, 0,
                                     _lib.current_stream_ptr(q.device))
    _lib.check(rc, "kitty_decode_attn_split")
    ml = ws.view(torch.float32)[:2 * H_Q].view(H_Q, 2).cpu().numpy()
    acc = ws[-(-2 * H_Q * 4 // 256) * 256:].view(torch.float32)[:H_Q * D].view(H_Q, D).double().cpu().numpy()
    assert (ml[:, 0] == 0).all()
    logits = (-2 * levels).astype(np.float32) * np.float32(scaling * np.float32(1.44269504088896340736))
    p = np.exp2(logits.astype(np.float64))
    # an fp32 exponential's unit in the last place and fp32 sums; what three fp16 numbers leave out below 2^-16
    bound = 3 * (p * 2.0 ** -22 + 2.0 ** -40)
    err = np.abs(acc[:, :len(own)] - 3 * p)
    assert (err <= bound).all(), (err / bound).max()
