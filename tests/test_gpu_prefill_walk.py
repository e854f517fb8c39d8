"""Chunked prefill: walks around the ring of 128 page addresses (staged 64 at a time), the loop for whole pages with
nothing, one, two and more of its tiles in front of the fp16 rows, and scalings that are negative or zero.

Tolerance: that of test_gpu_prefill.py, 2e-3 on fp16 outputs of size up to 4 (half an ulp of the output is 9.8e-4, the
probabilities' fp16 rounding about as much)."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv
from tests.test_gpu_prefill import ATOL, K, SC, _q, _run, _state  # noqa: F401 (K is a fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pages", [1, 3, 4, 5, 6, 31, 63, 64, 65, 95, 96, 97, 129, 200])
def test_walks_around_the_address_ring(K, pages):
    T0 = 32 + 128 * pages + 17
    cache, ol = _state(K, 1, 1, 4, T0, 0, T0 + 512, seed=pages)
    _run(K, cache, ol, 1, 4, 1, 70, seed=pages, what=f"{pages} pages")


@pytest.mark.parametrize("num_splits", [1, 2, 3, 7])
@pytest.mark.parametrize("pages", [70, 131])
def test_shares_around_the_address_ring(K, pages, num_splits):
    from kitty_amd.kvcache.kernels import kitty_attention as ka
    T0, Tq = 32 + 128 * pages + 90, 33
    cache, ol = _state(K, 1, 1, 4, T0, 0, T0 + 512, seed=pages)
    kc, vc = make_kv(1, 1, Tq, seed=pages + 1)
    q = _q(1, 4, Tq, pages)
    qd, kd, vd = (K.u.to_dev(x) for x in (q, kc, vc))
    out = torch.empty((1, Tq, 4, 128), dtype=torch.float16, device="cuda")
    need = ka._lib.lib().kitty_prefill_attn_workspace_bytes(1, 4, 128, Tq, num_splits)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda") if num_splits > 1 else None
    ka._launch_chunk(cache.kv_cache[0].descriptor(), qd, kd, vd, SC, out, ws, need, num_splits, "test")
    torch.cuda.synchronize()
    want = O.chunk_attention(ol, q, kc, vc, SC)
    assert np.abs(out.cpu().numpy().astype(np.float64) - want).max() <= ATOL


@pytest.mark.parametrize("T0", [0, 32 + 128 * 5 + 40])
@pytest.mark.parametrize("scaling", [-SC, 0.0])
def test_scalings_that_are_not_positive(K, T0, scaling):
    Tq = 150
    cache, ol = _state(K, 1, 2, 8, T0, 0, 2048, seed=T0 + 3)
    kc, vc = make_kv(1, 2, Tq, seed=4)
    q = _q(1, 8, Tq, 5)
    got, _ = K.pre(K.u.module(2, 8), K.u.to_dev(q), K.u.to_dev(kc), K.u.to_dev(vc), cache.kv_cache[0], scaling)
    torch.cuda.synchronize()
    want = O.chunk_attention(ol, q, kc, vc, scaling)
    assert np.abs(got.cpu().numpy().astype(np.float64) - want).max() <= ATOL
