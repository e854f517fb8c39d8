"""NaN and infinities in attention.  Head dimensions 64 and 256: a row one of whose logits is NaN or +inf comes out as 0, a logit of
-inf is a token that is not there - whichever wavefront, tile or share meets the token, and whatever else that one met.  Head dimension 128, chunks and prompts: such a row is NaN, in
one walk and in shares, and a prompt's rows in front of the token do not see it."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv

pytestmark = pytest.mark.gpu


def _state(D, T, seed):
    import kitty_amd
    from tests import gpu_util as u
    k, v = make_kv(2, 2, T, D=D, seed=seed)
    cache = kitty_amd.KittyCache(u.cfg(2, 4, D=D), 2, 2048)
    ol = O.OracleLayer(2, 2048, 2, D=D, D_BOOSTED=D // 4)
    cache.update(u.to_dev(k), u.to_dev(v), 0)
    cache.quantize_prefill(0)
    ol.update(k, v)
    ol.quantize_prefill()
    return u, cache.kv_cache[0], ol


def _query(D, T_q, seed):
    q = np.random.default_rng(seed).standard_normal((2, 4, T_q, D)).astype(np.float16)
    q[:, ::2, :, 0], q[:, 1::2, :, 0] = 1, -1         # even heads see +inf where a key's first channel is +inf, odd ones -inf
    return q


def _plant(L, ol, token, value):
    """Channel 0 of a key of (batch row 1, kv head 0) that lies in the sink or the Q-buffer."""
    sink = token < 32
    t = token if sink else (token - 32) % 128
    (L.Sink_Buffer_K if sink else L.Q_Buffer_K)[1, 0, t, 0] = value
    (ol.Sink_Buffer_K if sink else ol.Q_Buffer_K)[1, 0, t, 0] = value


def _expect(ref, value):
    """The oracle's result with the rows of (1, kv head 0) that meet a NaN or +inf logit set to 0."""
    ref = ref.copy()
    if np.isnan(value):
        ref[1, :, :2] = 0
    else:
        ref[1, :, 0] = 0                               # head 0 (+inf); head 1 sees -inf
    return ref


def _close(out, ref, what):
    got = out.float().cpu().numpy().astype(np.float64)
    assert np.isfinite(got).all() and (np.abs(got - ref) <= 2.0 ** -11 * np.abs(ref) + 2e-5).all(), what


# (tokens, the planted one): alone in its wavefront's share of the tile, with others, in the sink, in a tail tile
PLACES = [(3, 2), (9, 2), (32, 31), (35, 34), (32 + 128 + 3, 32 + 128 + 2), (32 + 256 + 70, 32 + 256 + 69), (32 + 256 + 70, 5)]


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T,token", PLACES)
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_decode(D, T, token, value):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    u, L, ol = _state(D, T, T)
    q = _query(D, 1, T)
    with np.errstate(all="ignore"):
        _plant(L, ol, token, value)
        ref = _expect(O.decode_attention(ol, q, D ** -0.5, reference_rounding=False, dequant="two"), value)
    out, _ = kitty_attention_forward(u.module(2, 4), u.to_dev(q), L, D ** -0.5, num_splits=1)
    _close(out, ref, (D, T, token))


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T,token", PLACES)
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("T_q", [1, 17])
def test_chunk(D, T, token, value, T_q, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import _lib
    from kitty_amd.kvcache.kernels import kitty_attention as A
    u, L, ol = _state(D, T, T)
    k, v = make_kv(2, 2, T_q, D=D, seed=T_q)
    q = _query(D, T_q, T)
    with np.errstate(all="ignore"):
        _plant(L, ol, token, value)
        ref = _expect(O.chunk_attention(ol, q, k, v, D ** -0.5, dequant="two"), value)
    for s in (1, 3, 20):
        monkeypatch.setattr(A, "_chunk_split_plan",
                            lambda *a, s=s: (s, _lib.lib().kitty_prefill_attn_workspace_bytes(2, 4, D, T_q, s)))
        out, _ = A.kitty_prefill_attention(u.module(2, 4), u.to_dev(q), u.to_dev(k), u.to_dev(v), L, D ** -0.5)
        _close(out, ref, (D, T, token, s))


@pytest.mark.parametrize("T,token", [(3, 2), (32, 31), (32 + 128 + 3, 32 + 128 + 2), (32 + 256 + 70, 5)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_chunk_128(T, token, value, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import _lib
    from kitty_amd.kvcache.kernels import kitty_attention as A
    u, L, ol = _state(128, T, T)
    k, v = make_kv(2, 2, 17, seed=17)
    q = _query(128, 17, T)
    with np.errstate(all="ignore"):
        _plant(L, ol, token, value)
        ref = _expect(O.chunk_attention(ol, q, k, v, 128 ** -0.5, dequant="two"), value)
    nan = np.zeros(ref.shape, bool)
    nan[1, :, :2 if np.isnan(value) else 1] = True
    for s in (1, 3, 20):
        monkeypatch.setattr(A, "_chunk_split_plan",
                            lambda *a, s=s: (s, _lib.lib().kitty_prefill_attn_workspace_bytes(2, 4, 128, 17, s)))
        out, _ = A.kitty_prefill_attention(u.module(2, 4), u.to_dev(q), u.to_dev(k), u.to_dev(v), L, 128 ** -0.5)
        got = out.float().cpu().numpy()
        assert (np.isnan(got) == nan).all(), s
        # fp16 probabilities (2^-11 each, relative) weigh rows of at most max|v|; half a unit of the fp16 result
        bound = 2.0 ** -11 * float(np.abs(v).max() + 4) + 2.0 ** -11 * np.abs(ref)
        assert (np.abs(got - ref)[~nan] <= bound[~nan]).all(), s


@pytest.mark.parametrize("T,token", [(5, 0), (40, 33), (300, 140), (700, 699)])
@pytest.mark.parametrize("shares", [1, 2, 5])
def test_prompt(T, token, shares, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd import _lib
    from kitty_amd.kvcache.kernels import kitty_attention as A
    from tests import gpu_util as u
    k, v = make_kv(1, 2, T, seed=T)
    k[0, 0, token, 3] = np.nan
    q = np.random.default_rng(T).standard_normal((1, 4, T, 128)).astype(np.float16)
    L = kitty_amd.KittyCache(u.cfg(2, 4), 1, 1024).kv_cache[0]
    qd, kd, vd = u.to_dev(q), u.to_dev(k), u.to_dev(v)
    monkeypatch.setattr(A, "_chunk_split_plan", lambda *a: (shares, _lib.lib().kitty_prefill_attn_workspace_bytes(1, 4, 128, T, shares)))
    assert A.prompt_attention_ready(qd, kd, vd, L)
    got = A.kitty_prompt_attention(qd, kd, vd, L, 128 ** -0.5)[0].float().cpu().numpy()      # [T, 4, 128]
    assert np.isnan(got[token:, :2]).all()
    clean = got.copy()
    clean[token:, :2] = 0
    assert np.isfinite(clean).all()
    k[0, 0, token, 3] = 0
    ref = np.concatenate([O.prefill_attention(q[0, 2 * h:2 * h + 2], k[0, h:h + 1], v[0, h:h + 1], 128 ** -0.5, 0) for h in (0, 1)])
    ref = ref.transpose(1, 0, 2)
    ref[token:, :2] = 0
    assert (np.abs(clean - ref) <= 2.0 ** -11 * np.abs(v).max() + 2.0 ** -11 * np.abs(ref)).all()


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("T,token", [(3, 1), (40, 31), (32 + 128 + 100, 32 + 128 + 60), (32 + 384, 32 + 20)])
@pytest.mark.parametrize("splits", [1, 3])
def test_infinite_values(D, T, token, splits):
    """A value that is infinite makes its channel infinite and no other: +-inf in fp16 rows; in packed pages a range so
    wide that the reference's fp16 arithmetic overflows (code * scale beyond 65504)."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import kitty_amd
    from kitty_amd.kvcache.kernels import kitty_attention_forward
    from tests import gpu_util as u
    k, v = make_kv(1, 2, T, D=D, seed=T)
    packed = token >= 32 and token < T - 128
    if packed:
        v[0, 0, token, ::2], v[0, 0, token, 1::2] = -60000, 60000
    else:
        v[0, 0, token, 3], v[0, 0, token, D - 2] = np.inf, -np.inf
    cache = kitty_amd.KittyCache(u.cfg(2, 4, D=D), 1, 2048)
    ol = O.OracleLayer(1, 2048, 2, D=D, D_BOOSTED=D // 4)
    with np.errstate(all="ignore"):
        cache.update(u.to_dev(k), u.to_dev(v), 0)
        cache.quantize_prefill(0)
        ol.update(k, v)
        ol.quantize_prefill()
        q = np.random.default_rng(T).standard_normal((1, 4, 1, D)).astype(np.float16)
        ref = O.decode_attention(ol, q, D ** -0.5, reference_rounding=False, dequant="two")
    assert (ol.PageCount_V * 128 > token - 32 >= 0) == packed and np.isinf(ref).any() and not np.isnan(ref).any()
    out, _ = kitty_attention_forward(u.module(2, 4), u.to_dev(q), cache.kv_cache[0], D ** -0.5, num_splits=splits)
    got = out.float().cpu().numpy().astype(np.float64)
    inf = np.isinf(ref)
    assert (got[inf] == ref[inf]).all()
    big = 60000 if packed else 8                            # fp32 sums over terms of that size
    assert (np.abs(got - ref)[~inf] <= 2.0 ** -11 * np.abs(ref[~inf]) + 2.5e-6 * big).all()
