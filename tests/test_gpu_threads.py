"""GPU: contexts of several threads share the page-locked pool and the store of series structures."""
import threading

import numpy as np
import pytest

from helpers import case, small_camera
from megamol_amd import SphereRenderer, _lib as L, params, scenes

pytestmark = pytest.mark.gpu


def passes(seed, times):
    """Frames and series of one context, larger and smaller ones in turn; their images."""
    out = []
    xyzr, rgba = scenes.random_spheres(3000 + 500 * seed, seed=seed, rmin=0.01, rmax=0.04)
    with SphereRenderer(0) as r:
        for k in range(times):
            w, h = ((120, 90), (333, 201), (64, 48))[(seed + k) % 3]
            r.set_spheres(xyzr, rgba)
            r.build(L.BUILD_REBUILD, 30)
            f = r.render(small_camera(w, h), params(w, h, spp=1 + k % 2, mode=L.MODE_AO, ao_distance=0.2))
            out += [f.rgba8, f.depth, f.hit_id]
            steps = 2 + (seed + k) % 3
            r.set_timesteps(np.stack([xyzr + np.float32(0.01 * t) * np.float32([1, 0, 0, 0]) for t in range(steps)]))
            p = params(w, h, spp=1, mode=L.MODE_LAMBERT)
            res, _ = r.render_batch([(t, small_camera(w, h), p) for t in range(steps)], refit_period=2, use_graph=bool(k % 2))
            out += [a for pair in res for a in pair]
    return out


def test_contexts_in_threads(gpu_renderer):
    """Four threads, each with a context of its own, get what they get one after the other."""
    case("contexts in threads")
    want = [[a.copy() for a in passes(s, 6)] for s in range(4)]
    got = [None] * 4

    def work(s):
        got[s] = passes(s, 6)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in range(4):
        assert got[s] is not None and len(got[s]) == len(want[s])
        for a, b in zip(got[s], want[s]):
            np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32))
