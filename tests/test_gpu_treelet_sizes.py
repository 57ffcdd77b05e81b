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
