"""GPU: treelets of every shape of their last levels: the device arrays equal the oracle's and frames
equal the brute-force oracle, for sphere counts about the sizes where a level, a wavefront's share of
the positions or a treelet ends, with equal, negative and zero coordinates."""
import numpy as np
import pytest

import oracle as O
from helpers import assert_frames_equal, case, oracle_params
from megamol_amd import _lib as L, look_at, params
from test_gpu_treelets import structure_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [256, 512, 1024])
@pytest.mark.parametrize("n", [2, 3, 4, 6, 7, 8, 14, 15, 16, 63, 64, 65, 127, 255, 256, 257, 511, 513, 767, 1023, 1026,
                               1031, 1279, 2047])
def test_ragged_treelets(gpu_renderer, M, n):
    r = gpu_renderer
    case(f"treelets M={M} n={n}")
    g = np.random.default_rng(n)
    xyzr = np.empty((n, 4), np.float32)
    xyzr[:, :3] = np.round(g.normal(size=(n, 3)) * 8) / 8  # many equal coordinates, zeros among them
    xyzr[::7, 1] = -0.0
    xyzr[:, 3] = g.uniform(0.02, 0.12, n)
    rgba = g.random((n, 4)).astype(np.float32)
    cam = look_at((0.1, 0.2, 6.0), (0, 0, 0), (0, 1, 0), 40.0, 33 / 25, 0.1, 20.0)
    try:
        r.set_option("accel", 1)
        r.set_option("treelet", M)
        r.set_spheres(xyzr, rgba)
        r.build(L.BUILD_REBUILD, 30)
        structure_equal(r.get_treelets(), O.Pkd(O.Bvh(xyzr, 30), M))
        for spp, mode in ((1, L.MODE_AO), (4, L.MODE_AO), (1, L.MODE_BOUNCE)):
            p = params(33, 25, spp=spp, mode=mode, ao_distance=1.0, max_bounces=2)
            f = r.render(cam, p)
            assert_frames_equal(f, O.render_brute(xyzr, rgba, cam, oracle_params(p)), what=f"M={M} n={n} spp={spp} mode={mode}")
    finally:
        r.set_option("accel", 0)
        r.set_option("treelet", 1024)


@pytest.mark.parametrize("size,window", [((1024, 640), None), ((1032, 640), None), ((1101, 733), None),
                                         ((1400, 900), (13, 7, 1177, 801)), ((2048, 1288), None)])
def test_frames_of_ordered_tiles(gpu_renderer, size, window):
    """Frames of two to eight tiles per wavefront take them in an order of their cost, which changes no
    pixel: at 10240 tiles of 8x8 (as they lie), just above, with ragged edges, in a window and past 40960
    (as they lie again), against the LBVH over the same spheres."""
    r = gpu_renderer
    w, h = size
    case(f"ordered tiles {size} {window}")
    g = np.random.default_rng(7)
    n = 6000
    xyzr = np.empty((n, 4), np.float32)
    xyzr[:, :3] = np.repeat(g.normal(size=(60, 3)) * 2, n // 60, 0) + g.normal(size=(n, 3)) * 0.15
    xyzr[:, 3] = g.uniform(0.005, 0.03, n)
    rgba = g.random((n, 4)).astype(np.float32)
    cam = look_at((0.3, 0.2, 9.0), (0, 0, 0), (0, 1, 0), 40.0, w / h, 0.1, 30.0)
    p = params(w, h, mode=L.MODE_AO, ao_distance=0.5, flags=L.FLAG_AUX)
    if window:
        p.window[:] = window
    frames = []
    try:
        for accel in (1, 0):
            r.set_option("accel", accel)
            r.set_option("treelet", 256)
            r.set_spheres(xyzr, rgba)
            r.build(L.BUILD_REBUILD, 30)
            frames.append(r.render(cam, p))
    finally:
        r.set_option("accel", 0)
        r.set_option("treelet", 1024)
    a, b = frames
    assert 0.02 < (b.hit_id >= 0).mean() < 0.9
    assert_frames_equal(a, {k: getattr(b, k) for k in ("hit_id", "t", "depth", "color", "rgba8", "aux")}, aux=True,
                        what=f"ordered tiles {size} {window}")
