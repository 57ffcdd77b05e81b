"""GPU: the packets that the rays of neighbouring pixels begin with part where the rays do."""
import numpy as np
import pytest

from helpers import assert_frames_equal, case
from megamol_amd import _lib as L, look_at, params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def clusters():
    """Small spheres in tight clusters: a pixel of a coarse image covers many, its neighbours others."""
    g = np.random.default_rng(2)
    n = 2_000_000
    centre = g.random((40, 3))
    xyzr = np.empty((n, 4), np.float32)
    xyzr[:, :3] = centre[np.sort(g.integers(0, 40, n))] + g.normal(size=(n, 3)) * 0.02
    xyzr[:, 3] = 0.0001
    return xyzr, g.random((n, 4)).astype(np.float32)


@pytest.mark.parametrize("spp", [2, 4, 16, 64])
@pytest.mark.parametrize("mode", [L.MODE_LAMBERT, L.MODE_AO])
def test_scattered_rays(gpu_renderer, clusters, mode, spp):
    """Frames whose rays part have the lane-per-pixel kernels' values bit for bit. A visit of a packet counts
    for all its lanes, and it goes on while the lanes that meet the visited nodes, less a quarter of all at
    each visit, have not used up a credit of 2048: so it makes at most 4 times the lane visits that meet
    something, and 4 x (2048 + 64) more; then each lane goes on by itself."""
    r = gpu_renderer
    r.set_spheres(*clusters)
    r.build(L.BUILD_REBUILD, 63)
    w, h = 317, 243
    cam = look_at((0.5, 0.5, 2.2), (0.5, 0.5, 0.5), (0, 1, 0), 40.0, w / h, 0.1, 10.0)
    p = params(w, h, spp=spp, mode=mode, ao_distance=0.1, flags=L.FLAG_AUX)
    frames, visits = [], []
    try:
        r.set_option("count_visits", 1)
        for lanes in (1, 0):
            case(f"scattered rays mode {mode} spp {spp} lanes {lanes}")
            r.set_option("sample_lanes", lanes)
            frames.append(r.render(cam, p))
            visits.append(r.counters()[0])
        r.set_option("count_visits", 0)
        r.set_option("sample_lanes", 1)
        frames.append(r.render(cam, p))
    finally:
        r.set_option("sample_lanes", 1)
        r.set_option("count_visits", 0)
    want = {k: getattr(frames[1], k) for k in ("hit_id", "t", "depth", "color", "rgba8", "aux")}
    assert (frames[1].hit_id >= 0).sum() > 1000
    for f in (frames[0], frames[2]):
        assert_frames_equal(f, want, aux=True, what=f"scattered rays mode {mode} spp {spp}")
    bound = 5 * visits[1] + 4 * 2112 * (-(-w // 8) * -(-h // 8) * spp)  # (packets of 64 rays)
    print(f"mode {mode} spp {spp}: {visits[0] / visits[1]:.2f} times the visits, {visits[0] / bound:.2f} of the bound")
    assert visits[0] <= bound
