"""The system of a particle, found by a table of every 256th: offsets on and beside the
table's steps, many systems within one, and a smaller forest after a larger one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(256, 256, 1, 255, 257), (255, 2, 254, 1, 513),
                                   (1,) * 300 + (3000,) + (2,) * 400, (70000, 1, 511, 100000),
                                   (1,) * 512 + (1,)])
def test_systems_stay_apart(bt, sizes):
    t = bt.Treecode(0.01, 0.5, 64)
    for sizes in (tuple(s + 300 for s in sizes), sizes):
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
        n = int(off[-1])
        pos, vel = bt.plummer(n, seed=99)
        t.alloc(n, off)
        t.ptcl_h2d(pos, vel)
        t.buildTree(16)
        t.computeMultipoles()
        t.makeGroups(5, 64)
        ids = t.ids(bt.ORDER_TREE)
        keys, perm = t.ph()
        by_tree = np.empty(n, np.uint64)
        by_tree[perm] = keys
        system = np.repeat(np.arange(len(sizes)), sizes)
        assert np.array_equal(system[ids], system)
        order = np.lexsort((np.arange(n), by_tree, system))
        assert np.array_equal(order, perm)
        groups = t.groups()
        assert np.array_equal(system[groups[:, 0]], system[groups.sum(1) - 1])
        assert np.array_equal(groups[:, 0], np.concatenate([[0], np.cumsum(groups[:, 1])[:-1]]))
    t.close()
