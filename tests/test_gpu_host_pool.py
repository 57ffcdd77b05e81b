"""GPU: what programs may do with the page-locked arrays that results arrive in: drop them, after an error
too, while the device is at work, hand them to forked workers, keep as many as they like."""
import gc
import os
import signal
import time

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


def test_sizes_change(gpu_renderer):
    """With one context idle blocks make room for those of another size at once."""
    case("host pool, another size")
    small = [L.host_empty((256 << 20,), np.uint8) for _ in range(4)]
    assert small[0].base is not None
    del small
    gc.collect()
    assert L.host_empty((600 << 20,), np.uint8).base is not None


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


def child_status(f, seconds=60):
    """Runs f in a forked child and returns the child's wait status (f returning true: 0)."""
    pid = os.fork()
    if pid == 0:
        code = 2
        try:
            code = 0 if f() else 1
        finally:
            os._exit(code)
    end = time.monotonic() + seconds
    while time.monotonic() < end:
        done, status = os.waitpid(pid, os.WNOHANG)
        if done:
            return status
        time.sleep(0.01)
    os.kill(pid, signal.SIGKILL)
    return os.waitpid(pid, 0)[1]


def test_frames_in_forked_children(gpu_renderer):
    """Worker processes forked from a renderer's read, write and drop its frames, as they can with any
    array, theirs forked in turn too; the parent's frames are not touched."""
    case("frames in forked children")
    xyzr, rgba = scenes.random_spheres(2000, seed=4, rmin=0.02, rmax=0.06)
    names = ("rgba8", "depth", "color", "t", "hit_id")
    with SphereRenderer(0) as r:
        r.set_spheres(xyzr, rgba)
        r.build()
        frames = [r.render(small_camera(w, h), params(w, h)) for w, h in ((64, 48), (333, 201), (64, 48))]
        dropped = r.render(small_camera(90, 70), params(90, 70))
        del dropped  # an idle block of the pool
        want = [{k: getattr(f, k).copy() for k in names} for f in frames]

        def equal():
            return all((getattr(f, k).view(np.uint32) == w[k].view(np.uint32)).all() for f, w in zip(frames, want)
                       for k in names)

        def child():
            ok = equal() and child_status(equal) == 0
            for f in frames:
                f.color[:] = 1.0
            frames.clear()
            gc.collect()
            return ok and L.host_empty((1 << 20,), np.uint8).base is None

        assert child_status(child) == 0
        assert equal()
        again = r.render(small_camera(64, 48), params(64, 48))
        np.testing.assert_array_equal(again.rgba8, want[0]["rgba8"])
        assert equal()


@pytest.mark.parametrize("mb,blocks", [(300, 1), (40, 20)])
def test_dropping_results_does_not_wait(busy, mb, blocks):
    """Arrays of any size, and many of them, are dropped at once while another renderer's frames are
    queued; only a renderer that must wait for its own buffers gives the memory back."""
    case(f"drop {blocks} x {mb} MB beside a busy renderer")
    held = [L.host_empty((mb << 20,), np.uint8) for _ in range(blocks)]
    assert held[0].base is not None
    gc.collect()  # (what other tests left; not part of the time below)
    long_work(busy)
    t0 = time.perf_counter()
    del held
    t1 = time.perf_counter()
    busy.sync()
    t2 = time.perf_counter()
    assert t1 - t0 < 0.5 * (t2 - t1), (t1 - t0, t2 - t1)


def test_idle_memory_is_given_back(gpu_renderer):
    """In use and idle together the pool takes 1 GB; past that arrays are ordinary until a device buffer
    grows, which leaves at most 256 MB idle."""
    case("idle memory of the host pool")
    del_me = [L.host_empty((256 << 20,), np.uint8) for _ in range(4)]
    assert any(a.base is not None for a in del_me)
    del del_me
    gc.collect()
    with SphereRenderer(0) as r:
        xyzr, rgba = scenes.random_spheres(2000, seed=4, rmin=0.02, rmax=0.06)
        r.set_spheres(xyzr, rgba)
        r.build()
        r.render_async(small_camera(64, 48), params(64, 48))
        assert L.host_empty((600 << 20,), np.uint8).base is None
        r.render_async(small_camera(640, 480), params(640, 480))
        r.sync()
        assert L.host_empty((600 << 20,), np.uint8).base is not None
