"""GPU: traversals whose stacks leave LDS, in every kernel: scenes of spheres so large that a ray meets both
children of nearly every node on its way down, so that the stack grows by an entry per level. How many
entries it holds at the first leaf is counted on the tree itself."""
import numpy as np
import pytest

import oracle as O
from helpers import assert_frames_equal, case, oracle_params, sample_ray, small_camera
from megamol_amd import _lib as L, params, scenes

pytestmark = pytest.mark.gpu

W, H = 21, 17
CAM = small_camera(W, H, pos=(0.5, 0.45, 2.4))


def pushes(box, child, o, d):
    """Entries pushed between the root and the first leaf of a ray that takes the nearer child."""
    node, count = 0, 0
    while node >= 0:
        tn = []
        for side in (0, 1):
            lo, hi = box[node, 6 * side:6 * side + 3].astype(np.float64), box[node, 6 * side + 3:6 * side + 6].astype(np.float64)
            a, b = (lo - o) / d, (hi - o) / d
            near, far = max(np.minimum(a, b).max(), 0.0), np.maximum(a, b).min()
            tn.append(near if near <= far else np.inf)
        if np.isinf(min(tn)):
            break
        count += not np.isinf(max(tn))
        node = child[node, 0] if tn[0] <= tn[1] else child[node, 1]
    return count


def most_pushes(box, child):
    return max(pushes(box, child, *sample_ray(CAM, W, H, x, y)) for x in range(0, W, 5) for y in range(0, H, 4))


def big_spheres(n, seed):
    xyzr, rgba = scenes.random_spheres(n, seed=seed, rmin=0.1, rmax=0.2)
    return xyzr, rgba


@pytest.mark.parametrize("stack,entries", [(8, 6), (16, 10)])
def test_lbvh_stacks_spill(gpu_renderer, stack, entries):
    r = gpu_renderer
    xyzr, rgba = big_spheres(30000, 3)
    r.set_spheres(xyzr, rgba)
    r.build(L.BUILD_REBUILD, 63)
    box, child, *_ = r.bvh()
    assert most_pushes(box, child) >= entries + 2  # (one entry is the bottom of the stack)
    try:
        r.set_option("stack_lds", stack)
        for mode, spp, refill, bounces in ((L.MODE_LAMBERT, 1, -1, 0), (L.MODE_AO, 1, 16, 0), (L.MODE_AO, 3, -1, 0),
                                           (L.MODE_AO, 16, -1, 0), (L.MODE_BOUNCE, 1, -1, 2)):
            what = f"spilled stacks {stack}: mode {mode} spp {spp} refill {refill} bounces {bounces}"
            case(what)
            r.set_option("refill", refill)
            p = params(W, H, spp=spp, mode=mode, ao_distance=0.01, max_bounces=bounces)
            o = O.render_brute(xyzr, rgba, CAM, oracle_params(p))
            for count in (0, 1):
                r.set_option("count_visits", count)
                assert_frames_equal(r.render(CAM, p), o, what=what)
            r.counters()
            assert r.get_option("stack_overflow") == 0
    finally:
        r.set_option("stack_lds", 16)
        r.set_option("refill", -1)
        r.set_option("count_visits", 0)


def test_treelet_stacks_spill(gpu_renderer):
    r = gpu_renderer
    xyzr, rgba = big_spheres(1 << 20, 4)
    try:
        r.set_option("accel", 1)
        r.set_option("treelet", 256)
        r.set_spheres(xyzr, rgba)
        r.build(L.BUILD_REBUILD, 63)
        t = r.get_treelets()
        assert most_pushes(t["top_box"], t["top_child"]) >= 12  # 10 entries in LDS, one of them the bottom
        for mode, spp in ((L.MODE_AO, 1), (L.MODE_LAMBERT, 2)):
            case(f"spilled treelet stacks: mode {mode} spp {spp}")
            p = params(W, H, spp=spp, mode=mode, ao_distance=0.01)
            r.set_option("count_visits", 1)
            assert_frames_equal(r.render(CAM, p), O.render_brute(xyzr, rgba, CAM, oracle_params(p)), what=f"treelets {mode}")
            r.counters()
            assert r.get_option("stack_overflow") == 0
    finally:
        r.set_option("accel", 0)
        r.set_option("treelet", 1024)
        r.set_option("count_visits", 0)
