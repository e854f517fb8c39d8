"""A prompt's values into the simulator's buffer in one launch against the copy and the pass in place: the same bits at
every edge of the range (no tail, a tail, one quantized token), for each group size, in both layouts of the source."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [161, 288, 289, 417, 1000])
@pytest.mark.parametrize("group,bits,sink,bitdec", [(128, 2, 32, False), (64, 4, 0, False), (32, 1, 5, True)])
@pytest.mark.parametrize("layout", ["token-major", "contiguous"])
def test_values_on_their_way_in(L, group, bits, sink, bitdec, layout):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from kitty_amd import sim
    g = torch.Generator().manual_seed(L + group)
    k, v = (torch.randn(2, L, 3, 128, generator=g).half().cuda().transpose(1, 2) for _ in range(2))
    if layout == "contiguous":
        k, v = k.contiguous(), v.contiguous()
    cfg = dict(sink_length=sink, group_size=group, vbits=bits, promote_ratio=0.25, VCache_BitDecoding=bitdec, PostQuant=False)
    outs = []
    for fused in (True, False):
        c = sim.KittyKVCache(sim.KittyKVCacheConfig(**cfg), max_length=L + 4)
        if not fused:
            c._values_from = lambda *a: False
        outs.append([x.clone() for x in c.update(k, v, 0)])
        outs[-1] += [x.clone() for x in c.update(k[:, :, :1], v[:, :, :1], 0)]
    for a, b in zip(*outs):
        assert torch.equal(a, b)
