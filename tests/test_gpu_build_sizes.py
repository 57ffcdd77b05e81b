"""GPU: the LBVH at the sizes where the build changes its kernels (one workgroup's sort up to 8192 or
16384 spheres, tiles of 8 or 16 keys per thread, one column launch or three, spans of 64 or 256
chunks), against the oracle's tree: keys, leaf order, references and boxes bit for bit."""
import numpy as np
import pytest

import oracle as O
from helpers import case
from megamol_amd import _lib as L
from test_gpu_parity import leaf_pair_form

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 63, 64, 65, 1024, 1025, 2048, 2049, 5120, 5121, 8192, 8193, 12288, 12289, 16384, 16385, 131073,
         524288, 524289, 2097152, 2097153]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("bits", [30, 63])
def test_tree_at_the_edges(gpu_renderer, n, bits):
    case(f"build n={n} bits={bits}")
    g = np.random.default_rng(n)
    xyzr = np.empty((n, 4), np.float32)
    xyzr[:, :3] = g.normal(size=(n, 3))
    xyzr[:, 3] = g.uniform(0.001, 0.01, n)
    if n > 100:
        xyzr[n // 3: n // 3 + 40, :3] = xyzr[5, :3]  # equal keys, ordered by index
    gpu_renderer.set_spheres(xyzr)
    gpu_renderer.build(L.BUILD_REBUILD, bits)
    _, bounds, _ = gpu_renderer.info()
    lo, hi = (xyzr[:, :3] - xyzr[:, 3:]).min(0), (xyzr[:, :3] + xyzr[:, 3:]).max(0)
    np.testing.assert_array_equal(bounds, np.concatenate([lo, hi]))
    box, child, ids, keys, height, pairs = gpu_renderer.bvh()
    ob = O.Bvh(xyzr, bits)
    obox, ochild, oids, okeys = ob.arrays()
    np.testing.assert_array_equal(keys, okeys)
    np.testing.assert_array_equal(ids, oids)
    if n == 1:
        return
    echild, epairs, stored = leaf_pair_form(ochild)
    np.testing.assert_array_equal(child[stored], echild[stored])
    np.testing.assert_array_equal(pairs[stored], epairs[stored])
    np.testing.assert_array_equal(box[stored].view(np.uint32), obox[stored].view(np.uint32))
    # a refit over moved spheres takes the same tree with their boxes
    moved = xyzr.copy()
    moved[:, :3] += g.normal(size=(n, 3)).astype(np.float32) * np.float32(0.01)
    gpu_renderer.set_spheres(moved)
    gpu_renderer.build(L.BUILD_REFIT, bits)
    rbox, rchild, _, _, _, _ = gpu_renderer.bvh()
    np.testing.assert_array_equal(rchild[stored], echild[stored])
    root = np.concatenate([np.minimum(rbox[0, 0:3], rbox[0, 6:9]), np.maximum(rbox[0, 3:6], rbox[0, 9:12])])
    np.testing.assert_array_equal(root, np.concatenate([(moved[:, :3] - moved[:, 3:]).min(0),
                                                        (moved[:, :3] + moved[:, 3:]).max(0)]))
