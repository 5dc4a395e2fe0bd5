"""Sorts of more than 2^17 keys leave out the lowest digits and order the runs of
equal leading digits in the gather; runs of more than 65 are sorted again by every
digit.  Either way: keys in order, ties in input order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 150001


def _check_orders(t, pos, off):
    n = len(pos)
    keys, perm = t.ph()
    assert np.array_equal(np.sort(perm), np.arange(n))
    by_tree = np.empty(n, np.uint64)
    by_tree[perm] = keys
    ids = t.ids(t_order_tree)
    tree_pos, _ = t.ptcl_d2h(t_order_tree)
    assert np.array_equal(pos[ids], tree_pos)
    same = (tree_pos[1:, :3] == tree_pos[:-1, :3]).all(1)
    same[off[1:-1] - 1] = False
    assert (ids[1:][same] > ids[:-1][same]).all()
    for b, e in zip(off[:-1], off[1:]):
        assert np.array_equal(np.sort(ids[b:e]), np.arange(b, e))
        assert np.array_equal(np.argsort(by_tree[b:e], kind="stable") + b, perm[b:e])


t_order_tree = 1


def _cluster(bt, n, members, spread):
    """A Plummer sphere of which `members` are within `spread` of one point."""
    pos, vel = bt.plummer(n, seed=51)
    rng = np.random.default_rng(5)
    k = rng.choice(n, members, replace=False)
    pos[k, :3] = np.float32(0.71) + (spread * rng.standard_normal((members, 3))).astype(np.float32)
    return pos, vel


# spread 1e-4: some tens share 13 digits of the box's 32; 0 and 1e-6: all of them do
@pytest.mark.parametrize("members,spread", [(2, 0.0), (64, 1e-6), (65, 1e-6), (66, 0.0),
                                            (5000, 1e-6), (40000, 1e-2), (1000, 1e-4)])
@pytest.mark.parametrize("fp64", [False, True])
def test_one_system(bt, oracle, members, spread, fp64):
    pos, vel = _cluster(bt, N, members, spread)
    real = np.float64 if fp64 else np.float32
    pos, vel = pos.astype(real), vel.astype(real)
    t = bt.Treecode(0.01, 0.5, 64, fp64=fp64)
    t.alloc(N)
    t.ptcl_h2d(pos, vel)
    for split in (5, 14):      # 14 digits of the groups' masks are past a short sort
        t.buildTree(16)
        t.computeMultipoles()
        t.makeGroups(split, 64)
        ids_now = t.ids(bt.ORDER_TREE)
        assert np.array_equal(np.sort(ids_now), np.arange(N))
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.computeMultipoles()
    t.makeGroups(5, 64)
    _check_orders(t, pos, np.array([0, N]))
    if not fp64:
        ref = oracle.reference_pipeline(pos, 16, 64, 0.5, 0.01, level_split=5)
        assert np.array_equal(t.tree(multipoles=False)["cells"], ref["tree"].cells)
        assert np.array_equal(t.groups(), ref["groups"])
    t.close()


# one, two system passes after the digits'
@pytest.mark.parametrize("nsys", [3, 300])
@pytest.mark.parametrize("members", [40, 400])
def test_forest(bt, nsys, members):
    rng = np.random.default_rng(nsys)
    off = np.sort(np.concatenate([[0, N], rng.choice(N - 1, nsys - 1, replace=False) + 1]))
    pos, vel = _cluster(bt, N, members, 1e-6)
    t = bt.Treecode(0.01, 0.5, 64)
    t.alloc(N, off.astype(np.int32))
    t.ptcl_h2d(pos, vel)
    t.buildTree(16)
    t.computeMultipoles()
    t.makeGroups(5, 64)
    _check_orders(t, pos, off)
    t.close()


@pytest.mark.parametrize("learned", [False, True])
def test_steps_into_a_cluster(bt, learned):
    """The drift of the first step brings 300 particles together: the step is
    finished with full sorts, eagerly and in a captured step, with equal results."""
    dt = 1.0 / 256
    pos, vel = _cluster(bt, N, 300, 1e-6)
    near = np.abs(pos[:, :3] - np.float32(0.71)).max(1) < 1e-4
    shift = np.random.default_rng(6).uniform(-0.2, 0.2, (int(near.sum()), 3))
    vel[near, :3] = (-shift / dt).astype(np.float32)
    pos[near, :3] += shift.astype(np.float32)
    out = []
    for graph in (False, True):
        t = bt.Treecode(0.05, 0.6, 64)
        t.alloc(N)
        t.ptcl_h2d(pos, vel)
        if learned:
            t.use_learned_theta(check_samples=0)
        t.buildTree(16)
        t.computeMultipoles()
        t.makeGroups(5, 64)
        t.computeForces()
        if graph:
            t.step_graph(dt, 16, 5, 64, nsteps=3)
            t.step_graph(dt, 16, 5, 64, nsteps=2)
        else:
            for _ in range(5):
                t.step(dt, 16, 5, 64)
        p, v = t.ptcl_d2h(bt.ORDER_INPUT)
        keys, _ = t.ph()
        assert (np.diff(keys.astype(np.int64)) >= 0).all()
        out.append((p, v, t.acc(bt.ORDER_INPUT), t.counts()))
        t.close()
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)
    assert out[0][3] == out[1][3]
    assert np.isfinite(out[0][2]).all()
