"""Forests of many small groups are walked by one wave per group, smaller ones by teams
of four: the forces are the same bits as, or other bits than, those of a context that is
told to walk by waves.  The interactions of the groups are equal either way."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsys,m,kind,split,waves", [
    (161, 815, "learned", 5, True), (160, 820, "learned", 5, False),
    (256, 512, "learned", 5, False), (2, 131073, "learned", 5, True),
    (161, 815, "fp64", 5, True), (256, 512, "fp64", 5, False),
    (256, 513, "fixed", 7, True), (256, 513, "fixed", 6, False), (257, 511, "fixed", 7, False)])
def test_forest_walks(bt, nsys, m, kind, split, waves):
    n = nsys * m
    pos, vel = bt.plummer(n, seed=77)
    fp64 = kind == "fp64"
    real = np.float64 if fp64 else np.float32
    t = bt.Treecode(0.01, 0.5, 64, fp64=fp64)
    t.alloc(n, np.arange(0, n + 1, m, dtype=np.int32))
    t.ptcl_h2d(pos.astype(real), vel.astype(real))
    if kind == "learned":
        t.use_learned_theta(check_samples=0)
    t.buildTree(16)
    t.computeMultipoles()
    t.makeGroups(split, 64)
    out = []
    for blocks_per_cu in (0, 8):
        t.set_walk_options(blocks_per_cu=blocks_per_cu)
        t.computeForces()
        out.append((t.acc(bt.ORDER_PH), t.group_counts()))
    t.close()
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0]) == waves
    a, b = (o[0].astype(np.float64) for o in out)
    assert np.linalg.norm(a - b) <= (1e-13 if fp64 else 1e-6) * np.linalg.norm(b)
