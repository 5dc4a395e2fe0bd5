"""The longest runs of equal leading key digits that are put in order without a sort by
every digit, and the first that are not: keys in order, ties in input order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 4000: a tile in LDS; 150001: radix passes, the gather orders the runs
@pytest.mark.parametrize("n", [4000, 150001])
@pytest.mark.parametrize("members", [255, 256, 257, 258])
@pytest.mark.parametrize("spread", [0.0, 1e-6])
def test_run_lengths(bt, n, members, spread):
    pos, vel = bt.plummer(n, seed=95)
    rng = np.random.default_rng(7)
    k = rng.choice(n, members, replace=False)
    pos[k, :3] = np.float32(0.71) + (spread * rng.standard_normal((members, 3))).astype(np.float32)
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
    assert np.array_equal(pos[ids], tree_pos)
    same = (tree_pos[1:, :3] == tree_pos[:-1, :3]).all(1)
    assert (ids[1:][same] > ids[:-1][same]).all()
    by_tree = np.empty(n, np.uint64)
    by_tree[perm] = keys
    assert np.array_equal(np.argsort(by_tree, kind="stable"), perm)
