"""GPU: the traversal's branches at the sizes and directions where they can go wrong, bit for bit
against the brute-force oracle: rays of one pixel that lie in several octants (no packet walk),
axis-parallel rays, trees of one to five leaves (the second sphere of the last leaf), equal-t ties
and deep trees whose stacks leave LDS."""
import numpy as np
import pytest

import oracle as O
from helpers import assert_frames_equal, case, oracle_params
from megamol_amd import _lib as L, look_at, params, scenes

pytestmark = pytest.mark.gpu


def check(r, xyzr, rgba, cam, p, what, **opts):
    case(what)
    try:
        for k, v in opts.items():
            r.set_option(k, v)
        r.set_spheres(xyzr, rgba)
        r.build(L.BUILD_REBUILD, 63)
        g = r.render(cam, p)
    finally:
        r.set_option("stack_lds", 16)
        r.set_option("leaf_pairs", 1)
        r.set_option("refill", -1)
    o = O.render_brute(xyzr, rgba, cam, oracle_params(p))
    assert_frames_equal(g, o, what=what)
    return o


@pytest.mark.parametrize("spp", [1, 2, 16, 64])
@pytest.mark.parametrize("direction", [(0, 0, -1), (1, 0, 0), (0, -1, 0.001), (-1, -1, -1)])
def test_octant_seams(gpu_renderer, direction, spp):
    """Looking along an axis the image centre divides the octants, inside pixels too (odd sizes)."""
    xyzr, rgba = scenes.random_spheres(4000, seed=31, rmin=0.005, rmax=0.03)
    xyzr[100:110] = xyzr[50]
    d = np.array(direction, np.float64)
    w, h = (33, 25) if spp == 64 else (65, 49)
    cam = look_at(tuple(0.5 - 1.6 * d / np.linalg.norm(d)), (0.5, 0.5, 0.5), (0, 1, 0) if direction[1] != -1 else (0, 0, 1),
                  40.0, w / h, 0.1, 10.0)
    p = params(w, h, spp=spp, mode=L.MODE_AO, ao_distance=0.3)
    o = check(gpu_renderer, xyzr, rgba, cam, p, f"octants {direction} spp {spp}")
    assert (o["hit_id"] >= 0).mean() > 0.2


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("spp", [1, 64])
@pytest.mark.parametrize("mode", [L.MODE_LAMBERT, L.MODE_AO])
def test_few_leaves(gpu_renderer, n, spp, mode):
    xyzr, rgba = scenes.random_spheres(n, seed=n, lo=0.3, hi=0.7, rmin=0.1, rmax=0.2)
    cam = look_at((0.5, 0.5, 2.2), (0.5, 0.5, 0.5), (0, 1, 0), 40.0, 17 / 13, 0.1, 10.0)
    p = params(17, 13, spp=spp, mode=mode, ao_distance=1.0)
    for pairs in (1, 0):
        check(gpu_renderer, xyzr, rgba, cam, p, f"{n} leaves spp {spp} mode {mode} pairs {pairs}", leaf_pairs=pairs)


@pytest.mark.parametrize("spp", [1, 3, 64])
@pytest.mark.parametrize("refill", [-1, 0, 16])
def test_deep_tree_small_stack(gpu_renderer, spp, refill):
    """Spheres whose distances shrink geometrically make a deep tree (63-bit codes); with 4 entries
    in LDS its stacks spill."""
    g = np.random.default_rng(5)
    n = 3000
    s = 0.5 ** (np.arange(n) % 20 * 0.9)
    xyzr = np.empty((n, 4), np.float32)
    xyzr[:, :3] = 0.5 + (g.random((n, 3)) - 0.5) * s[:, None]
    xyzr[:, 3] = 0.01 * s + 1e-5
    rgba = g.random((n, 4)).astype(np.float32)
    cam = look_at((0.52, 0.47, 1.4), (0.5, 0.5, 0.5), (0, 1, 0), 30.0, 1.0, 0.1, 10.0)
    p = params(21, 21, spp=spp, mode=L.MODE_AO, ao_distance=0.5)
    check(gpu_renderer, xyzr, rgba, cam, p, f"deep tree spp {spp} refill {refill}", stack_lds=8, refill=refill)
    gpu_renderer.set_option("count_visits", 1)
    try:
        gpu_renderer.render(cam, p)
        gpu_renderer.counters()
        assert gpu_renderer.get_option("stack_overflow") == 0
    finally:
        gpu_renderer.set_option("count_visits", 0)


@pytest.mark.parametrize("w,h", [(1, 1), (8, 8), (9, 1), (3, 70), (130, 67)])
@pytest.mark.parametrize("blocks", [8, 1])
def test_work_queues(gpu_renderer, w, h, blocks):
    """Every pixel is rendered whatever the number of tiles is beside the 8 queues and the
    wavefronts: fewer tiles than queues, tiles divided into units (64 samples), all wavefronts' first
    units and many more."""
    xyzr, rgba = scenes.random_spheres(1500, seed=3, rmin=0.02, rmax=0.06)
    cam = look_at((0.5, 0.5, 2.0), (0.5, 0.5, 0.5), (0, 1, 0), 40.0, w / h, 0.1, 10.0)
    try:
        gpu_renderer.set_option("blocks_per_cu", blocks)
        for spp in (1, 2, 64) if w * h < 2000 else (1, 2):
            for refill in (0, 16):
                p = params(w, h, spp=spp, mode=L.MODE_AO, ao_distance=0.3)
                check(gpu_renderer, xyzr, rgba, cam, p, f"queues {w}x{h} spp {spp} refill {refill} blocks {blocks}",
                      refill=refill)
    finally:
        gpu_renderer.set_option("blocks_per_cu", 8)


@pytest.mark.parametrize("spp", [2, 4, 16, 64, 192])
@pytest.mark.parametrize("window", [None, (3, 5, 13, 11)])
def test_passes_without_a_hit(gpu_renderer, spp, window):
    """A few spheres on a wide background: whole passes that miss (they end early where a pass is the
    pixel) next to pixels hit by some of their samples, over two accumulated frames and with the window
    at an odd offset, against the lane-per-pixel kernels bit for bit."""
    r = gpu_renderer
    xyzr, rgba = scenes.random_spheres(40, seed=41, rmin=0.01, rmax=0.06)
    w, h = 29, 23
    cam = look_at((0.5, 0.5, 2.5), (0.5, 0.5, 0.5), (0, 1, 0), 50.0, w / h, 0.1, 10.0)
    frames = {}
    try:
        r.set_spheres(xyzr, rgba)
        r.build(L.BUILD_REBUILD, 30)
        for lanes in (1, 0):
            r.set_option("sample_lanes", lanes)
            for k in range(2):
                case(f"missed passes spp {spp} window {window} lanes {lanes} frame {k}")
                p = params(w, h, spp=spp, mode=L.MODE_AO, ao_distance=0.3, frame_idx=k, accumulate=1,
                           background=(0.2, 0.3, 0.4, 0.5), flags=L.FLAG_AUX)
                if window:
                    p.window[:] = window
                frames[lanes, k] = r.render(cam, p)
    finally:
        r.set_option("sample_lanes", 1)
    for k in range(2):
        a, b = frames[1, k], frames[0, k]
        hit = b.hit_id >= 0
        assert 0 < hit.sum() < 0.5 * hit.size
        assert_frames_equal(a, {n: getattr(b, n) for n in ("hit_id", "t", "depth", "color", "rgba8", "aux")}, aux=True,
                            what=f"missed passes spp {spp} window {window} frame {k}")


@pytest.mark.parametrize("mode,bounces", [(L.MODE_LAMBERT, 0), (L.MODE_AO, 0), (L.MODE_BOUNCE, 1), (L.MODE_BOUNCE, 4)])
def test_frames_about_the_small_size(gpu_renderer, mode, bounces):
    """One sample: a small frame against the oracle, and a frame one tile row above 7680 tiles of 8x8
    against a window of exactly that many."""
    r = gpu_renderer
    xyzr, rgba = scenes.random_spheres(3000, seed=51, rmin=0.01, rmax=0.05)
    cam = lambda w, h: look_at((0.5, 0.5, 2.2), (0.5, 0.5, 0.5), (0, 1, 0), 40.0, w / h, 0.1, 10.0)
    p = params(61, 47, mode=mode, max_bounces=bounces, ao_distance=0.3)
    check(r, xyzr, rgba, cam(61, 47), p, f"mode {mode} bounces {bounces} small frame")
    w, h = 1024, 488
    case(f"mode {mode} bounces {bounces} {w}x{h} and window")
    p = params(w, h, mode=mode, max_bounces=bounces, ao_distance=0.3, flags=L.FLAG_AUX)
    a = r.render(cam(w, h), p)
    p.window[:] = (0, 0, w, 480)
    b = r.render(cam(w, h), p)
    assert_frames_equal(b, {k: getattr(a, k)[:480] for k in ("hit_id", "t", "depth", "color", "rgba8", "aux")}, aux=True,
                        what=f"mode {mode} bounces {bounces} window")
