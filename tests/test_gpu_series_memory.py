"""GPU: the device memory that a batched series leaves behind for later ones."""
import numpy as np
import pytest

from helpers import case
from megamol_amd import SphereRenderer, _lib as L, look_at, params

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

KEPT = 1 << 30    # what the library says it keeps at most
SLACK = 64 << 20  # rounding of some dozen allocations
CAM = look_at((50, 70, 270), (50, 50, 50), (0, 1, 0), 40.0, 64 / 48, 1.0, 1000.0)


def series(r, steps, n):
    xs = np.empty((steps, n, 4), np.float32)
    xs[..., :3] = np.random.default_rng(n).random((1, n, 3)) * 100.0
    xs[..., 3] = 0.4
    r.set_timesteps(xs)


def used(r, steps):
    """Device memory in use after a series, without any kept structures of its own and with them."""
    p = params(64, 48, spp=1, mode=L.MODE_AO, ao_distance=1.5)
    out = []
    for one in (0, 1):
        r.set_option("batch_launch", one)
        r.render_batch([(t, CAM, p) for t in range(steps)], refit_period=steps)
        free, total = torch.cuda.mem_get_info()
        out.append(total - free)
    return out


def test_kept_structures_are_bounded(gpu_renderer):
    """A series whose structures take 1.7 GB leaves at most 1 GB of them allocated, and a second
    renderer's series uses these instead of keeping as much again."""
    case("series memory")
    steps, n = 8, 3_000_000
    assert (steps - 1) * n * 80 > KEPT + 2 * SLACK
    with SphereRenderer(0) as a, SphereRenderer(0) as b:
        series(a, steps, n)
        plain, kept = used(a, steps)
        assert kept - plain <= KEPT + SLACK, (plain, kept)
        series(b, steps, n)
        plain_b, kept_b = used(b, steps)
        assert kept_b - plain_b <= SLACK, (plain_b, kept_b)
    free, total = torch.cuda.mem_get_info()
    assert total - free <= plain, "destroyed contexts keep nothing"
