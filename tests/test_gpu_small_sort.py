"""The two-launch sort of small systems: keys in order, ties in input order, and
the tree order it gives equal to the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a tile holds 4096 pairs, 32 tiles are the most this sort takes
@pytest.mark.parametrize("n", [2, 63, 65, 4095, 4096, 4097, 8193, 40000, 131072, 131073])
@pytest.mark.parametrize("twins", [False, True])
def test_small_sorts(bt, oracle, n, twins):
    pos, vel = bt.plummer(n, seed=11)
    if twins:      # every other particle on the point of one of three others, across the tiles
        pos[1::2, :3] = pos[np.arange(n)[1::2] % min(3, n), :3]
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(n)
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    ids = t.ids(bt.ORDER_TREE)
    tree_pos, _ = t.ptcl_d2h(bt.ORDER_TREE)
    t.computeMultipoles()
    t.makeGroups(5, 64)
    keys, perm = t.ph()
    t.close()
    ref = oracle.reference_pipeline(pos, 16, 64, 0.5, 0.01, level_split=5)
    assert np.array_equal(tree_pos, ref["pos_tree"])
    assert np.array_equal(pos[ids], tree_pos)
    same = (tree_pos[1:, :3] == tree_pos[:-1, :3]).all(1)
    assert (ids[1:][same] > ids[:-1][same]).all()          # ties in input order
    by_tree = np.empty(n, np.uint64)
    by_tree[perm] = keys
    assert np.array_equal(np.argsort(by_tree, kind="stable"), perm)
