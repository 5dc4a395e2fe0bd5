"""The cell build's tiles hold 256 particles up to 2^17 and 1024 above: the edges of
both against the oracle, in a context that is allocated for a larger system first."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [255, 256, 257, 512, 131071, 131072, 131073])
@pytest.mark.parametrize("nleaf", [16, 64])
def test_cells_after_a_larger_system(bt, oracle, n, nleaf):
    pos, vel = bt.plummer(n, seed=71)
    ref = oracle.reference_pipeline(pos, nleaf, 64, 0.5, 0.01, level_split=5)
    t = bt.Treecode(0.01, 0.5, 64)
    big, bvel = bt.plummer(140000, seed=72)
    t.alloc(len(big))
    t.ptcl_h2d(big, bvel)
    t.buildTree(nleaf)
    t.alloc(n)
    t.ptcl_h2d(pos, vel)
    t.buildTree(nleaf)
    t.computeMultipoles()
    got = t.tree()
    t.close()
    assert np.array_equal(got["cells"], ref["tree"].cells)
