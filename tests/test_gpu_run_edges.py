"""Runs of equal leading key digits at the edges of the loops that put them in order (8
keys one by one, then 8 at a time; 16 others in a tile, 256 after radix passes), at the
ends of the arrays and of a forest's systems: keys in order, ties in input order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(bt, pos, off):
    n = len(pos)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(n, off)
    t.ptcl_h2d(pos, np.zeros_like(pos))
    t.buildTree(16)
    ids = t.ids(bt.ORDER_TREE)
    tree_pos, _ = t.ptcl_d2h(bt.ORDER_TREE)
    t.computeMultipoles()
    t.makeGroups(5, 64)
    keys, perm = t.ph()
    t.close()
    assert np.array_equal(pos[ids], tree_pos)
    off = np.array([0, n]) if off is None else off
    same = (tree_pos[1:, :3] == tree_pos[:-1, :3]).all(1)
    same[off[1:-1] - 1] = False
    assert (ids[1:][same] > ids[:-1][same]).all()
    by_tree = np.empty(n, np.uint64)
    by_tree[perm] = keys
    for b, e in zip(off[:-1], off[1:]):
        assert np.array_equal(np.sort(ids[b:e]), np.arange(b, e))
        assert np.array_equal(np.argsort(by_tree[b:e], kind="stable") + b, perm[b:e])


# at: where in the key order the run lies (the box's corners are its ends)
@pytest.mark.parametrize("n", [1000, 4000, 40000, 150001])
@pytest.mark.parametrize("members", [8, 9, 10, 15, 16, 17, 18, 25, 257])
@pytest.mark.parametrize("at", [-15.9, 0.71, 15.9])
def test_runs(bt, n, members, at):
    pos, _ = bt.plummer(n, seed=29)
    pos[:, :3] = np.clip(pos[:, :3], -15.0, 15.0)
    rng = np.random.default_rng(members)
    k = rng.choice(n, members, replace=False)
    pos[k, :3] = np.float32(at) + (1e-5 * rng.standard_normal((members, 3))).astype(np.float32)
    _check(bt, pos, None)


# one and two system passes; every system has a run, half of them one of `members` + 1,
# and neighbouring systems' runs lie at the same point
@pytest.mark.parametrize("nsys", [7, 300])
@pytest.mark.parametrize("members", [1, 8, 16, 256, 400])
def test_runs_of_systems(bt, nsys, members):
    n = 150001
    off = (np.arange(nsys + 1) * (n // nsys)).astype(np.int32)
    off[-1] = n
    pos, _ = bt.plummer(n, seed=31)
    pos[:, :3] = np.clip(pos[:, :3], -15.0, 15.0)
    rng = np.random.default_rng(nsys)
    for s in range(nsys):
        m = members + s % 2
        k = off[s] + rng.choice(off[s + 1] - off[s], m, replace=False)
        at = np.float32((-15.9, 15.9)[s // 2 % 2])
        pos[k, :3] = at + (1e-5 * rng.standard_normal((m, 3))).astype(np.float32)
    _check(bt, pos, off)
