"""Boxes and sizes of the linear BVH where its refit can go wrong: trees inside
one workgroup's 1024 primitives, at its edge and over several, with leaves of
one triangle, of a few, and of more triangles than a workgroup has; node for
node the oracle's tree."""
import numpy as np
import pytest

from firefly_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_prims", [1, 8, 1500])
@pytest.mark.parametrize("n", [2, 1023, 1024, 1025, 2048, 5000])
def test_refit_equals_oracle(gpu, oracle, n, max_prims):
    rng = np.random.default_rng(n)
    pos = (rng.uniform(-1, 1, (n, 1, 3)) + rng.normal(scale=0.05, size=(n, 3, 3))).astype(np.float32)
    mats = np.zeros((1, abi.FF_MAT_FLOATS), np.float32)
    mats[0, 0] = abi.FF_MAT_DIFFUSE
    mats[0, 10:14] = -1
    nrm = np.tile(np.array([0, 1, 0], np.float32), (n, 3, 1))
    sc = abi.Scene(gpu, pos, nrm, None, np.zeros(n, np.int32), mats, max_prims=max_prims, builder=abi.FF_BVH_LBVH)
    nodes, ordered = sc.bvh()
    want_nodes, want_ordered = oracle.lbvh_build(pos, max_prims)
    assert np.array_equal(ordered, want_ordered)
    assert nodes.tobytes() == want_nodes.tobytes()
    sc.close()
