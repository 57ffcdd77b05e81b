"""GPU: what programs may do with the page-locked arrays that results arrive in: drop them, after an error
too, while the device is at work."""
import gc

import numpy as np
import pytest

from helpers import case, small_camera
from megamol_amd import SphereRenderer, _lib as L, params, scenes

pytestmark = pytest.mark.gpu


def long_work(r, frames=8):
    """Queues some 100 ms of frames of this renderer and returns at once."""
    p = params(1920, 1080, spp=64, mode=L.MODE_AO, ao_distance=0.1)
    for _ in range(frames):
        r.render_async(small_camera(1920, 1080), p)


@pytest.fixture(scope="module")
def busy():
    with SphereRenderer(0) as r:
        xyzr, rgba = scenes.random_spheres(1_000_000, seed=4, rmin=0.002, rmax=0.004)
        r.set_spheres(xyzr, rgba)
        r.build()
        long_work(r, 1)  # buffers are allocated now
        r.sync()
        yield r


def test_refused_download_leaves_no_copy_behind(busy):
    """A download that is refused (features of a frame rendered without them) has queued nothing: the
    arrays of the failed call are free for others, here filled while its renderer is still at work."""
    case("refused download")
    n = 1920 * 1080
    long_work(busy)
    with pytest.raises(L.MMHRTError, match="no aux buffer"):
        busy.download(1920, 1080, aux=True)
    gc.collect()
    blocks = [L.host_empty((n * k,), np.uint32) for k in (1, 1, 4, 1, 1, 4)]
    for b in blocks:
        b[:] = 0x5A5A5A5A
    busy.sync()
    for b in blocks:
        assert (b == 0x5A5A5A5A).all()
    f = busy.download(1920, 1080, outputs=("depth", "hit_id"))
    assert (f.hit_id >= 0).any() and np.isfinite(f.depth).all()
