"""Dense causal attention of a prompt on the chunk kernel (what the hook runs on an empty layer) against float64, and
the calls that have to stay with torch's attention."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


def _setup(B, T, H_Q, H, layout):
    from kitty_amd import hf
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=128, num_key_value_heads=H, num_attention_heads=H_Q, hidden_size=H_Q * 128)
    g = torch.Generator().manual_seed(T + H_Q)

    def make(n):
        x = torch.randn(B, T, n, 128, generator=g).half().cuda().transpose(1, 2)
        return x if layout == "token-major" else x.contiguous()
    return hf, hf.KittyHFCache(cfg, B, T + 256), make(H_Q), make(H), make(H)


@pytest.mark.parametrize("T", [1, 31, 129, 257, 700])
@pytest.mark.parametrize("H_Q,H,layout", [(2, 2, "token-major"), (8, 2, "contiguous"), (24, 2, "token-major"), (8, 8, "token-major"), (8, 4, "contiguous")])
def test_prompt_attention(T, H_Q, H, layout):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    hf, cache, q, k, v = _setup(2, T, H_Q, H, layout)
    mod = types.SimpleNamespace(layer_idx=0)
    kk, vv = cache.update(k, v, 0)
    assert hf.prompt_attention_ready(q, kk, vv, cache.kv_cache[0])
    out, _ = hf.kitty_attention(mod, q, kk, vv, None, scaling=128 ** -0.5)
    assert out.shape == (2, T, H_Q, 128) and out.is_contiguous() and cache.get_seq_length(0) == T
    qd, kd, vd = (x.double().cpu() for x in (q, k, v))
    ref = torch.nn.functional.scaled_dot_product_attention(qd, kd.repeat_interleave(H_Q // H, 1), vd.repeat_interleave(H_Q // H, 1),
                                                           is_causal=True, scale=128 ** -0.5).transpose(1, 2)
    # fp16 probabilities (2^-11 each, relative) weigh rows of at most max|v|; half a unit of the fp16 result
    bound = 2.0 ** -11 * float(vd.abs().max()) + 2.0 ** -11 * ref.abs()
    assert ((out.double().cpu() - ref).abs() <= bound).all()


def test_what_stays_with_torch():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    hf, cache, q, k, v = _setup(1, 40, 4, 2, "token-major")
    L = cache.kv_cache[0]
    ready = hf.prompt_attention_ready
    assert ready(q, k, v, L)
    assert not ready(q.float(), k, v, L) and not ready(q, k[:, :1], v[:, :1], L) and not ready(q[:, :3], k, v, L)
    assert not ready(q, k, v.contiguous(), L) and not ready(q, k.cpu(), v.cpu(), L) and not ready(q[:, :, :39], k, v, L)
    assert not ready(torch.nn.Parameter(q), k, v, L) and not ready(q.clone().requires_grad_(), k, v, L)
    wide = torch.zeros(1, 4, 40, 132, device="cuda", dtype=torch.float16)[..., :128]
    assert not ready(wide, k, v, L)
    with torch.no_grad():
        assert ready(q.clone().requires_grad_().detach(), k, v, L)
    kk, vv = cache.update(k, v, 0)                              # gradients flow as before
    qg = q.clone().requires_grad_()
    out, _ = hf.kitty_attention(types.SimpleNamespace(layer_idx=0), qg, kk, vv, None, scaling=128 ** -0.5)
    out.float().sum().backward()
    assert torch.isfinite(qg.grad).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_autocast_gives_the_result_its_type(dtype):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    hf, cache, q, k, v = _setup(1, 40, 4, 2, "token-major")
    with torch.autocast("cuda", dtype=dtype):
        kk, vv = cache.update(k, v, 0)
        out, _ = hf.kitty_attention(types.SimpleNamespace(layer_idx=0), q, kk, vv, None, scaling=128 ** -0.5)
        ref = torch.nn.functional.scaled_dot_product_attention(q, k.repeat_interleave(2, 1), v.repeat_interleave(2, 1), is_causal=True,
                                                               scale=128 ** -0.5).transpose(1, 2)
    assert out.dtype == ref.dtype == dtype and torch.equal(out, ref) and cache.get_seq_length(0) == 40
