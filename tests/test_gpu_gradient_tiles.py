"""GPU: the 16-block tiles of the data-gradient kernel (taken from 512 workgroups on) at every level and
width of the network, over images whose last tiles are partial in each of its three tile shapes, against
the 4-block tiles that a single image takes."""
import numpy as np
import pytest

from helpers import case
from megamol_amd import denoiser as D
from test_denoiser_cpu import random_features

pytestmark = pytest.mark.gpu

LEVEL = [0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0, 0, 0]


def tile(w, h):
    """The tile shape that covers the image with the fewest pixels, the widest on a tie."""
    shapes = [(64, 4), (32, 8), (16, 16)]
    return min(shapes, key=lambda s: -(-w // s[0]) * s[0] * (-(-h // s[1]) * s[1]))


@pytest.mark.parametrize("h,w,shapes", [(72, 120, [(64, 4), (64, 4), (32, 8), (16, 16)]),
                                        (120, 72, [(16, 16), (16, 16), (32, 8), (16, 16)]),
                                        (72, 88, [(32, 8), (64, 4), (32, 8), (16, 16)])])
def test_sixteen_block_tiles(gpu_renderer, h, w, shapes):
    """1024 copies of one image have its gradients: the loss is a mean, 2^-10 scales every bf16 gradient
    exactly and the kernels round each pixel's gradient alike, so only the order of the fp32 sums over
    1024 x more pixels differs: 2^-24 times the square root of 8.8 million terms is 1.8e-4. One column of
    wrong gradients would be a hundred times that."""
    n = 1024
    assert [tile(w >> k, h >> k) for k in range(4)] == shapes
    assert all((w >> k) % s[0] or (h >> k) % s[1] for k, s in enumerate(shapes))
    large = []
    for l, (name, c1, c2, co, _) in enumerate(D.LAYERS):
        blocks = (c1 + c2) // 16
        groups = 1 if blocks <= 5 else 2
        px = (h >> LEVEL[l]) * (w >> LEVEL[l])
        assert px // 256 * groups < 512, "the single image takes the small tiles"
        if l > 0 and n * px // 256 * groups >= 512:
            large.append(name)
    assert len(large) >= 13, large
    case(f"denoiser gradients, {n} copies of {h}x{w}")
    d = D.Denoiser(gpu_renderer, seed=7)
    feats = random_features(1, h, w, seed=h + w)
    target = np.random.default_rng(8).random((1, h, w, 3)).astype(np.float32)
    _, one = d.train_step(feats, target, 2.0, lr=0.0, apply=False, want_grads=True)
    _, many = d.train_step(np.repeat(feats, n, 0), np.repeat(target, n, 0), 2.0, lr=0.0, apply=False, want_grads=True)
    for (name, *_), (w1, b1), (wn, bn) in zip(D.LAYERS, D.split_params(one), D.split_params(many)):
        a, b = np.append(w1, b1), np.append(wn, bn)
        assert np.linalg.norm(b - a) < 2e-4 * np.linalg.norm(a), (name, np.linalg.norm(b - a) / np.linalg.norm(a))
        print(f"{name}: {np.linalg.norm(b - a) / np.linalg.norm(a):.1e}")
