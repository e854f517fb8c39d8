"""``update`` of one decode token on the GPU (one launch, kitty_append_row) against the slice copies the same
method makes on a CPU cache, step by step: sink fill, ring fill, ring wrap, both Q-buffers filling up."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


def _source(kind, B, H, D, gen):
    if kind == "token-major":                      # a projection's layout
        return torch.randn(B, 1, H, D, generator=gen).half().transpose(1, 2)
    if kind == "odd offset":                       # rows that do not start on 16 bytes: copied first
        return torch.randn(B * H * D + 3, generator=gen).half()[3:].view(B, H, 1, D)
    if kind == "bfloat16":                         # converted, as a slice assignment converts
        return torch.randn(B, H, 1, D, generator=gen).bfloat16()
    return torch.randn(B, H, 1, D, generator=gen).half()


@pytest.mark.parametrize("D,H,B", [(64, 1, 1), (64, 3, 2), (128, 8, 1), (128, 33, 2), (256, 9, 3)])
@pytest.mark.parametrize("kind", ["contiguous", "token-major", "odd offset", "bfloat16"])
def test_rows_land_where_the_slice_copies_put_them(D, H, B, kind):
    from kitty_amd import KittyCache
    cfg = types.SimpleNamespace(num_hidden_layers=1, head_dim=D, num_key_value_heads=H, num_attention_heads=H,
                                hidden_size=H * D)
    gpu, cpu = KittyCache(cfg, B + 1, 1024), KittyCache(cfg, B + 1, 1024, device="cpu")
    gen = torch.Generator().manual_seed(D + H)
    a, b = gpu.kv_cache[0], cpu.kv_cache[0]
    names = ("Sink_Buffer_K", "Sink_Buffer_V", "Q_Buffer_K", "Q_Buffer_V", "Local_Buffer_V")
    # (sink, K rows waiting, V rows waiting, ring rows, ring head): around every edge of the state machine
    for sink, rk, rv, lv, off in ((1, 0, 0, 0, 0), (31, 0, 0, 0, 0), (32, 0, 0, 0, 0), (32, 127, 0, 127, 0),
                                  (32, 0, 0, 128, 0), (32, 5, 127, 128, 127), (32, 127, 126, 128, 64)):
        for L in (a, b):
            (L.Sink_Count, L.Q_Buffer_Count_K, L.Q_Buffer_Count_V, L.Local_Count_V, L.Write_Offset_Local_V) = \
                (sink, rk, rv, lv, off)
        for _ in range(2 if rk < 126 and rv < 126 else 1):
            k, v = _source(kind, B, H, D, gen), _source(kind, B, H, D, gen)
            kd, vd = k.cuda(), v.cuda()
            if kind == "odd offset":
                kd, vd = (torch.cat([x.new_zeros(3), x.flatten()])[3:].view(B, H, 1, D) for x in (kd, vd))
                assert kd.data_ptr() % 16
            assert gpu.update(kd, vd, 0) is False and cpu.update(k, v, 0) is False
        assert a.counts() == b.counts()
        for n in names:
            assert torch.equal(getattr(a, n).cpu(), getattr(b, n)), (n, sink, rk, rv, lv, off)
    a.Q_Buffer_Count_K = 128                       # a skipped flush is an error on the host, as in the reference
    with pytest.raises(AssertionError):
        gpu.update(kd, vd, 0)
