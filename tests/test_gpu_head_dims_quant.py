"""The quantizers at head dimensions 64 and 256: the ends of the boost range, token-major and single-page sources, pages that
take no boosted rows, bit for bit against the oracle; and NaN among the inputs, which takes no part in a group's range and
gets its largest code (plain fp32 arithmetic, every operation correctly rounded on both sides: no tolerance)."""
import numpy as np
import pytest
import torch

from oracle import kitty_oracle as O
from tests.helpers import make_kv

pytestmark = pytest.mark.gpu
CASES = [(64, 0, 1, False), (64, 64, 3, True), (64, 16, 9, True), (256, 0, 2, True), (256, 255, 1, False), (256, 64, 5, True)]


def _buffers(n, H, D, DB):
    return (torch.zeros((n, H * (32 * (D + DB) + D)), dtype=torch.uint8, device="cuda"),
            torch.zeros((n, H, D, 2), dtype=torch.float16, device="cuda"),
            torch.zeros((n, H * 32 * D), dtype=torch.uint8, device="cuda"),
            torch.zeros((n, H, 128, 2), dtype=torch.float16, device="cuda"))


@pytest.mark.parametrize("D, DB, pages, token_major", CASES)
def test_pages_bit_exact(D, DB, pages, token_major):
    from kitty_amd.kvcache.kernels import quantize_pack_k, quantize_pack_v
    B, H = 2, 3
    x, _ = make_kv(B, H, 5 + 128 * pages + 3, D=D, seed=D + DB, student_t=True)
    x[:, :, ::7] *= np.float16(0.0)                       # zeros of both signs among the ties
    pt = np.random.default_rng(DB).permutation(B * pages).reshape(B, pages).astype(np.int64)
    xd = torch.from_numpy(x).cuda()
    if token_major:
        xd = xd.transpose(1, 2).contiguous().transpose(1, 2)
    kc, km, vc, vm = _buffers(B * pages, H, D, DB)
    ptd = torch.from_numpy(pt).cuda()
    quantize_pack_k(xd, 5, pages, ptd, 0, kc, km, 128, DB)
    quantize_pack_v(xd, 5, pages, ptd, 0, vc, vm, 128)
    want = [np.zeros(tuple(t.shape), np.uint8 if t.dtype == torch.uint8 else np.float16) for t in (kc, km, vc, vm)]
    O.quantize_pack_k(x, 5, pages, pt, 0, want[0], want[1], 128, DB)
    O.quantize_pack_v(x, 5, pages, pt, 0, want[2], want[3], 128)
    for got, w in zip((kc, km, vc, vm), want):
        g = got.cpu().numpy()
        assert np.array_equal(g, w)   # (a zero minimum may have either sign)


@pytest.mark.parametrize("D", [64, 256])
def test_nan_leaves_the_range_and_takes_the_largest_code(D):
    from kitty_amd.kvcache.kernels import quantize_pack_k, quantize_pack_v, select_boost_k
    DB = D // 4
    g = torch.Generator().manual_seed(D)
    x = torch.randn(128, D, generator=g).half()
    bad = [3, 11, D - 2]
    for i, c in enumerate(bad):
        x[5 + 40 * i, c] = float("nan")
    x[:, bad[1]] = float("nan")                           # a channel of nothing else
    xd = x.cuda().view(1, 1, 128, D)
    pt = torch.zeros((1, 1), dtype=torch.int64, device="cuda")
    kc, km, vc, vm = _buffers(1, 1, D, DB)
    quantize_pack_k(xd, 0, 1, pt, 0, kc, km, 128, DB)
    quantize_pack_v(xd, 0, 1, pt, 0, vc, vm, 128)
    slots = select_boost_k(xd, 0, 1, 128, DB).view(D).cpu()
    assert [int(slots[c]) for c in bad] == [0, 1, 2]      # a NaN saturates the score: first, by channel

    def codes(v, qmax):                                   # groups along dim 0
        f = v.float()
        mn = torch.where(f.isnan(), torch.inf, f).amin(0)
        mx = torch.where(f.isnan(), -torch.inf, f).amax(0)
        scale = (mx - mn) / qmax
        scale = torch.where(scale < 1e-6, torch.tensor(1e-6), scale)
        t = (f - mn) / scale + 0.5
        return torch.where(t.isnan(), qmax, torch.minimum(t, qmax + 0.5).floor()).int(), scale.half(), mn.half()

    boosted = slots < DB
    want, scale, zero = codes(x, torch.where(boosted, 15.0, 3.0))
    plane = kc.view(-1)[:32 * D].view(D, 32).cpu()
    shift = 2 * torch.arange(4)
    lo = (plane.unsqueeze(-1).int() >> shift & 3).reshape(D, 128).t()
    rows = kc.view(-1)[32 * D:32 * (D + DB)].view(DB, 32).cpu()
    hi = (rows.unsqueeze(-1).int() >> shift & 3).reshape(DB, 128).t()
    got = lo.clone()
    got[:, boosted] += 4 * hi[:, slots[boosted].long()]
    assert torch.equal(got, want)
    m = km.view(D, 2).cpu()
    assert torch.equal(m[:, 0], scale) and torch.equal(m[:, 1], zero)

    want, scale, zero = codes(x.t(), torch.full((128,), 3.0))
    got = (vc.view(128, D // 4).cpu().unsqueeze(-1).int() >> shift & 3).reshape(128, D).t()
    assert torch.equal(got, want)
    m = vm.view(128, 2).cpu()
    assert torch.equal(m[:, 0], scale) and torch.equal(m[:, 1], zero)
