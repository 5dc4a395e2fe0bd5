"""Small sorts: pairs of a tile whose leading key digits agree are placed among each
other, and a tile in which more than 64 agree is sorted by every digit.  Keys in
order, ties in input order, and the tree order equal to the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 1, 8 and 9 tiles of 1024 pairs, 2048, 16 of 2048, and of 4096
@pytest.mark.parametrize("n", [1000, 8192, 8193, 32768, 32769])
@pytest.mark.parametrize("members,spread", [(2, 0.0), (64, 1e-5), (66, 1e-5), (900, 1e-5),
                                            (900, 0.0), (700, 1e-2)])
def test_runs_in_tiles(bt, oracle, n, members, spread):
    pos, vel = bt.plummer(n, seed=61)
    rng = np.random.default_rng(6)
    k = rng.choice(n, members, replace=False)
    pos[k, :3] = np.float32(0.37) + (spread * rng.standard_normal((members, 3))).astype(np.float32)
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
    assert (ids[1:][same] > ids[:-1][same]).all()
    by_tree = np.empty(n, np.uint64)
    by_tree[perm] = keys
    assert np.array_equal(np.argsort(by_tree, kind="stable"), perm)
