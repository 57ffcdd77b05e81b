"""GPU: a build option that is asked for is taken as it is, at its default's value too; without a request the
library adapts it to the scene's size. The tree is the same."""
import numpy as np
import pytest

from helpers import case
from megamol_amd import _lib as L, scenes

pytestmark = pytest.mark.gpu


def reached(child):
    """Mask of the nodes that the tree stores (leaf pairs leave gaps)."""
    m = np.zeros(len(child), bool)
    front = np.array([0])
    while len(front):
        m[front] = True
        c = child[front].ravel()
        front = c[c >= 0]
    return m


def test_requested_build_options_are_taken(gpu_renderer):
    r = gpu_renderer

    def build(n, bits, **opts):
        case(f"build options n={n} bits={bits} {opts}")
        for k, v in opts.items():
            r.set_option(k, v)
        r.set_spheres(scenes.random_spheres(n, seed=n)[0])
        r.build(L.BUILD_REBUILD, bits)
        box, child, ids, keys, _, _ = r.bvh()
        m = reached(child)
        return (r.get_option("used_sort_ri"), r.get_option("used_build_span")), (m, box[m], child[m], ids, keys)

    try:
        for n, bits, adapted in ((9_000, 30, 0), (9_000, 63, 8), (70_000, 30, 8), (600_000, 63, 16)):
            used, want = build(n, bits, sort_ri=-1, build_span=-1)
            assert used[0] == adapted and used[1] > 0
            assert r.get_option("sort_ri") == 16 and r.get_option("build_span") == 256
            for ri, span in ((16, 256), (8, 128), (32, 32), (16, 1)):
                used, got = build(n, bits, sort_ri=ri, build_span=span)
                assert used == (16 if ri == 32 and bits == 63 else ri, span)
                for a, b in zip(got, want):
                    np.testing.assert_array_equal(a.view(np.uint8), b.view(np.uint8))
            used, _ = build(n, bits, build_span=0)
            assert used[1] == 0
    finally:
        r.set_option("sort_ri", -1)
        r.set_option("build_span", -1)


@pytest.mark.parametrize("n,span", [(1000, 256), (66_000, 256), (256 * 1024, 256), (256 * 1024 + 1, 64),
                                    (1_000_000, 64)])
def test_spans_of_small_scenes(gpu_renderer, n, span):
    """Up to 256 chunks one span merges the straddlers, in builds and refits (spans of 64 chunks and the
    pass over their exports took 66 to 260 chunks 5 to 27 % longer)."""
    r = gpu_renderer
    case(f"spans n={n}")
    r.set_option("build_span", -1)
    r.set_spheres(scenes.random_spheres(n, seed=1)[0])
    for policy in (L.BUILD_REBUILD, L.BUILD_REFIT):
        r.set_option("used_build_span", 0)
        r.build(policy, 30)
        assert r.get_option("used_build_span") == span
