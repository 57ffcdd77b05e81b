"""GPU: the LBVH where the number of chunks changes the spans that merge the straddlers (one span up to
256 chunks, spans of 64 up to 8192, of 256 beyond), with chunks of 256 leaves, against the oracle's tree:
keys, leaf order, references and boxes bit for bit."""
import numpy as np
import pytest

import oracle as O
from helpers import case
from megamol_amd import _lib as L
from test_gpu_parity import leaf_pair_form

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks,span", [(256, 256), (257, 64), (8192, 64), (8193, 256)])
@pytest.mark.parametrize("bits", [30, 63])
def test_tree_at_the_span_edges(gpu_renderer, chunks, span, bits):
    r = gpu_renderer
    n = 256 * chunks if chunks % 256 == 0 else 256 * (chunks - 1) + 1  # the last chunk full, or of one leaf
    case(f"spans of {chunks} chunks, n={n} bits={bits}")
    g = np.random.default_rng(n)
    xyzr = np.empty((n, 4), np.float32)
    xyzr[:, :3] = g.normal(size=(n, 3))
    xyzr[:, 3] = g.uniform(0.001, 0.01, n)
    xyzr[n // 3: n // 3 + 40, :3] = xyzr[5, :3]  # equal keys, ordered by index
    try:
        r.set_option("build_chunk", 256)
        r.set_option("build_span", -1)
        r.set_spheres(xyzr)
        r.build(L.BUILD_REBUILD, bits)
        assert r.get_option("used_build_span") == span
        trees = [r.bvh()]
        r.build(L.BUILD_REFIT, bits)
        trees.append(r.bvh())
    finally:
        r.set_option("build_chunk", 1024)
    obox, ochild, oids, okeys = O.Bvh(xyzr, bits).arrays()
    echild, epairs, stored = leaf_pair_form(ochild)
    for box, child, ids, keys, height, pairs in trees:
        np.testing.assert_array_equal(keys, okeys)
        np.testing.assert_array_equal(ids, oids)
        np.testing.assert_array_equal(child[stored], echild[stored])
        np.testing.assert_array_equal(pairs[stored], epairs[stored])
        np.testing.assert_array_equal(box[stored].view(np.uint32), obox[stored].view(np.uint32))
