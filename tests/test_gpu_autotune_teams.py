"""A tuned context walks small systems by teams as an untuned one does: the forces of
the two are the same bits (those of one wave per group are summed in another order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,fp64", [(2000, False), (30000, False), (20011, True)])
def test_tuned_walk_is_the_default_walk(bt, n, fp64):
    pos, vel = bt.plummer(n, seed=23)
    real = np.float64 if fp64 else np.float32
    t = bt.Treecode(0.01, 0.5, 64, fp64=fp64)
    t.alloc(n)
    t.ptcl_h2d(pos.astype(real), vel.astype(real))
    best, rows = t.autotune(5)
    assert best["blocks_per_cu"] in (4, 8, 12, 16) and len(rows) == 13
    u = bt.Treecode(0.01, 0.5, 64, fp64=fp64)
    u.alloc(n)
    u.ptcl_h2d(*t.ptcl_d2h(bt.ORDER_INPUT))
    out = []
    for c in (t, u):
        c.buildTree(best["nleaf"])
        c.computeMultipoles()
        c.makeGroups(5, best["ncrit"])
        c.computeForces()
        out.append((c.acc(bt.ORDER_INPUT), c.walk_stack_max()))
    u.set_walk_options(blocks_per_cu=best["blocks_per_cu"])   # by hand: a wave per group
    u.computeForces()
    waves = u.acc(bt.ORDER_INPUT)
    t.close()
    u.close()
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    assert not np.array_equal(out[0][0], waves)
