"""GPU: the page-locked arrays that frames are downloaded into, and the structures a batched series
keeps between calls."""
import ctypes as C
import gc

import numpy as np
import pytest

from helpers import case, small_camera
from megamol_amd import SphereRenderer, _lib as L, look_at, params, scenes

pytestmark = pytest.mark.gpu


def test_frames_own_their_memory(gpu_renderer):
    """A frame keeps its values while later frames of the same size are rendered, and after the frames
    before it are gone; its arrays are writable and contiguous, and outlive their renderer."""
    case("frames in page-locked memory")
    xyzr, rgba = scenes.random_spheres(2000, seed=4, rmin=0.02, rmax=0.06)
    with SphereRenderer(0) as r:
        r.set_spheres(xyzr, rgba)
        r.build()
        cams = [small_camera(90, 70, pos=(0.5, 0.5, 2.0 + 0.1 * i)) for i in range(4)]
        frames, copies = [], []
        for c in cams:
            frames.append(r.render(c, params(90, 70)))
            copies.append([getattr(frames[-1], k).copy() for k in ("rgba8", "depth", "color", "t", "hit_id")])
        del frames[1]
        gc.collect()
        r.render(cams[0], params(90, 70))
        a = frames[0].color
        assert a.flags.writeable and a.flags.c_contiguous and a.dtype == np.float32 and a.shape == (70, 90, 4)
    for f, want in zip(frames, (copies[0], copies[2], copies[3])):
        for k, w in zip(("rgba8", "depth", "color", "t", "hit_id"), want):
            np.testing.assert_array_equal(getattr(f, k).view(np.uint32), w.view(np.uint32))
        f.color[:] = 0.0


def test_host_pool(gpu_renderer):
    """Blocks do not overlap, foreign pointers are refused, and past the pool's bound arrays are ordinary."""
    case("host pool")
    lib = L.load()
    sizes = [1, 4096, 16384, 16385, 1 << 20, (1 << 20) + 1]
    ptr = []
    for n in sizes:
        p = C.c_void_p()
        assert lib.mmhrt_host_alloc(n, C.byref(p)) == L.OK
        ptr.append(p.value)
    for p, n in sorted(zip(ptr, sizes)):
        for q in ptr:
            assert q <= p or q >= p + n
    p = C.c_void_p()
    assert lib.mmhrt_host_alloc(2 << 30, C.byref(p)) == L.E_OOM and not p.value
    assert lib.mmhrt_host_alloc(0, C.byref(p)) == L.E_INVALID
    for q in ptr:
        assert lib.mmhrt_host_free(q) == L.OK
    assert lib.mmhrt_host_free(ptr[0]) == L.E_INVALID
    held = [L.host_empty((1 << 28,), np.uint8) for _ in range(5)]
    held[4][-1] = 7
    assert held[4].base is None and held[0].base is not None
    del held
    gc.collect()
    a = L.host_empty((1 << 28,), np.uint8)
    assert a.base is not None


@pytest.mark.parametrize("accel", [0, 1])
def test_series_of_changing_sizes(gpu_renderer, accel):
    """Series of more and fewer timesteps and spheres one after the other, over the structures kept from
    the call before, equal single renders."""
    g = np.random.default_rng(9)
    cam = look_at((10, 14, 55), (10, 10, 10), (0, 1, 0), 40.0, 64 / 48, 1.0, 200.0)
    p = params(64, 48, spp=1, mode=L.MODE_AO, ao_distance=1.5)
    with SphereRenderer(0) as r:
        r.set_option("accel", accel)
        for steps, n, period, graph in ((3, 4000, 2, True), (6, 9000, 3, False), (2, 700, 1, True), (6, 9000, 4, True)):
            case(f"series accel {accel}: {steps} x {n}, period {period}, graph {graph}")
            xs = np.empty((steps, n, 4), np.float32)
            xs[..., :3] = g.random((steps, n, 3)) * 20.0
            xs[..., 3] = 0.4
            r.set_timesteps(xs)
            out, _ = r.render_batch([(t, cam, p) for t in range(steps)], refit_period=period, use_graph=graph)
            for t in range(steps):
                r.set_spheres(xs[t])
                r.build(L.BUILD_REBUILD, 30)
                f = r.render(cam, p, outputs=("rgba8", "depth"))
                np.testing.assert_array_equal(out[t][0], f.rgba8)
                np.testing.assert_array_equal(out[t][1].view(np.uint32), f.depth.view(np.uint32))
