"""Decode attention at head dimensions 64 and 256 on either side of the line between its two kernels (a tile shared by four wavefronts, and a
page per wavefront): with a tile a compute unit, two, and walks of as many tiles as the former still takes, in the default number of
splits; and the latter's group sizes and high planes in batches of short walks."""
import numpy as np
import pytest
import torch

from tests.helpers import make_kv
from tests.test_gpu_head_dims_pages import _check, _layer

pytestmark = pytest.mark.gpu


def _run(D, B, H_KV, G, T, splits, boosted=None):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    k, v = make_kv(B, H_KV, T, D=D, seed=T + G)
    u, cache, ol = _layer(D, B, H_KV, H_KV * G, k, v, boosted)
    q = np.random.default_rng(G).standard_normal((B, H_KV * G, 1, D)).astype(np.float16)
    _check(u, cache, ol, q, D, H_KV, G, splits, f"D={D} B={B} T={T} G={G}")


# walks x tiles: 256, 257; 512, 516; 2 x 64, 2 x 65; 12 x 24, 12 x 25 (256 compute units)
@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("B,H_KV,tiles", [(64, 2, 2), (257, 1, 1), (128, 1, 4), (129, 1, 4), (5, 1, 64), (5, 1, 65), (12, 1, 24), (12, 1, 25)])
def test_line(D, B, H_KV, tiles):
    _run(D, B, H_KV, 2, 32 + 128 * (tiles - 1) - (9 if tiles > 1 else 1), (None, 1))


@pytest.mark.parametrize("D", [64, 256])
@pytest.mark.parametrize("G,T", [(1, 32 + 128 * 4), (5, 32 + 128 * 5 + 127), (6, 32 + 128 * 4 + 1), (16, 32 + 128 * 5 + 64)])
def test_pages_of_short_walks(D, G, T):
    _run(D, 131, 1, G, T, (None, 1, 2, 9))


@pytest.mark.parametrize("D,boosted", [(64, 0), (64, 32), (256, 0), (256, 80)])
def test_high_planes_of_short_walks(D, boosted):
    _run(D, 131, 1, 4, 32 + 128 * 4 + 40, (None, 1), boosted)
