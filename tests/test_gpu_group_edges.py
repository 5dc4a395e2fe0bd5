"""makeGroups at the edges of its tiles and words: group lists equal to chunks of
NCRIT cut from the runs of masked keys, per system."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expected(keys, off, level_split, ncrit):
    masked = keys >> np.uint64(63 - 3 * level_split)
    n = len(keys)
    start = np.ones(n, bool)
    start[1:] = masked[1:] != masked[:-1]
    start[off[:-1]] = True
    begins = np.flatnonzero(start)
    ends = np.append(begins[1:], n)
    out = [(b, min(ncrit, e - b)) for r0, e in zip(begins, ends) for b in range(r0, e, ncrit)]
    return np.array(out, np.int32)


def _check(bt, pos, vel, off, level_split, ncrit):
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(len(pos), off if len(off) > 2 else None)
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.makeGroups(level_split, ncrit)
    keys, perm = t.ph()
    got = t.groups()
    ids = t.ids(bt.ORDER_PH)
    assert np.array_equal(ids, t.ids(bt.ORDER_TREE)[perm])
    t.close()
    assert np.array_equal(got, _expected(keys, off, level_split, ncrit))


# a tile holds 1024 particles in words of 64; a run may start many tiles earlier
@pytest.mark.parametrize("level_split,ncrit", [(1, 64), (1, 7), (5, 64), (7, 48), (21, 1)])
@pytest.mark.parametrize("n", [2, 64, 65, 1023, 1025, 4096, 70001])
def test_groups_of_one_system(bt, n, level_split, ncrit):
    pos, vel = bt.plummer(n, seed=17)
    _check(bt, pos, vel, np.array([0, n], np.int32), level_split, ncrit)


@pytest.mark.parametrize("sizes", [(1, 63, 64, 65, 1023, 1, 2049), (40000, 3, 30000)])
def test_groups_of_a_forest(bt, sizes):
    n = sum(sizes)
    pos, vel = bt.plummer(n, seed=18)
    _check(bt, pos, vel, np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32), 2, 48)


def test_one_run_over_many_tiles(bt):
    """All but one particle in one octant: its run starts 60 tiles before the last
    and its length is no multiple of NCRIT."""
    n = 61441
    pos, vel = bt.plummer(n, seed=19)
    pos[:, :3] = 5.0 + 0.01 * pos[:, :3]
    pos[0, :3] = -50.0
    _check(bt, pos, vel, np.array([0, n], np.int32), 3, 48)
