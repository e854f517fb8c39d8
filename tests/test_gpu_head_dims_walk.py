"""Chunked prefill at head dimensions 64 and 256: whole packed tiles in a loop of their own in front of, behind and between the
tiles with fp16 rows, in one share and in several; blocks of 32 and of 48 rows at D = 64, and their remainders.

Tolerance: 2e-3 as in test_gpu_head_dims.py (half an ulp of an output of up to 4 is 9.8e-4; the probabilities are fp32 numbers)."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv
from tests.test_gpu_head_dims import ATOL, K, _q  # noqa: F401 (K is a fixture)

pytestmark = pytest.mark.gpu


# (D, G, T0, T_q): T0 ends inside a page, on a page, on the ring's edge; G and T_q give two or three column tiles at D = 64
@pytest.mark.parametrize("D,G,T0,Tq", [(64, 4, 32 + 128 * 6 + 50, 8), (64, 4, 32 + 128 * 6, 50), (64, 7, 32 + 128 * 3 + 127, 13),
                                       (64, 16, 32 + 128 * 2, 5), (64, 1, 32 + 128 * 4 + 1, 140), (256, 4, 32 + 128 * 5 + 50, 9),
                                       (256, 16, 32 + 128 * 3, 3), (256, 1, 20, 131), (256, 2, 32 + 128 * 2 + 127, 30)])
def test_chunk_shares(K, D, G, T0, Tq):
    from kitty_amd.kvcache.kernels import kitty_attention as ka
    B, H = 2, 1
    k, v = make_kv(B, H, T0 + Tq, D=D, seed=D + T0)
    cache = K.KittyCache(K.u.cfg(H, G, D=D), B, 2048)
    cache.update(K.u.to_dev(k[:, :, :T0]), K.u.to_dev(v[:, :, :T0]), 0)
    cache.quantize_prefill(0)
    ol = O.OracleLayer(B, 2048, H, D=D, D_BOOSTED=D // 4)
    ol.update(k[:, :, :T0], v[:, :, :T0])
    ol.quantize_prefill()
    q, kc, vc = _q(B, G, Tq, D, T0), k[:, :, T0:], v[:, :, T0:]
    want = O.chunk_attention(ol, q, kc, vc, D ** -0.5, dequant="two")
    qd, kd, vd = (K.u.to_dev(x) for x in (q, kc, vc))
    lib = ka._lib.lib()
    for shares in (1, 2, 3, 5):
        out = torch.empty((B, Tq, G, D), dtype=torch.float16, device="cuda")
        need = lib.kitty_prefill_attn_workspace_bytes(B, G, D, Tq, shares)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda") if shares > 1 else None
        ka._launch_chunk(cache.kv_cache[0].descriptor(), qd, kd, vd, D ** -0.5, out, ws, need, shares, "test")
        torch.cuda.synchronize()
        err = np.abs(out.cpu().numpy().astype(np.float64) - want).max()
        assert err <= ATOL, (shares, err)
